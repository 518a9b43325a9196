// Merge of the per-work-group partial rows a point-streaming kernel wrote
// and, for a whole iteration, the FP64 divide and the centroid shift: one
// kernel, launched after the streaming kernel on the same stream.
//
// (A variant that merged inside the streaming kernel, with the last
// work-group to arrive doing the work, was measured slower on gfx950: every
// work-group's agent-scope release fence writes back the XCD's L2, which
// holds the freshly written labels, and same-address device atomics take
// about 45 ns each.)
#pragma once

#include "clk_common.hpp"

namespace clk {

// A partial row holds nv = d + mass value rows of k values, [nv][k]: the d
// feature sums, then (mass) the cluster masses in the same type.
template <typename In, typename MassT, typename CenT>
struct MergeArgs {
    const In *part = nullptr;  // [rows][nv][k]
    uint32_t rows = 0;
    uint32_t d = 0;
    uint64_t k = 0;
    bool mass = false;
    double *sums = nullptr;     // [d][k]
    MassT *masses = nullptr;    // [k]
    bool divide = false;        // overwrite sums / masses and write centroids; else accumulate
    CenT *centroids = nullptr;  // divide: [d][k]
    const CenT *old_centroids = nullptr;  // divide: for the shift (may be null)
    // divide: receives the shift (may be null); must hold 0 when the merge
    // starts (the streaming kernel before it writes the 0)
    double *max_shift = nullptr;
    uint32_t lanes = 0, clusters = 0;  // set by launch_merge
};

using MergeF32 = MergeArgs<double, uint32_t, float>;
using MergeF64 = MergeArgs<double, uint64_t, double>;
using MergeU32 = MergeArgs<uint32_t, uint32_t, float>;  // masses only

template <typename In, typename MassT, typename CenT>
int launch_merge(clk_context *ctx, MergeArgs<In, MassT, CenT> a, const char *name, hipStream_t stream);

// sums[i] += the column sums of part[rows][count].
inline int launch_merge_sums(clk_context *ctx, const double *part, uint64_t rows, uint64_t count, double *sums,
                             hipStream_t stream)
{
    MergeF32 m;
    m.part = part;
    m.rows = (uint32_t)rows;
    m.d = 1;
    m.k = count;
    m.sums = sums;
    return launch_merge(ctx, m, "ReduceVectorParcol", stream);
}

}  // namespace clk
