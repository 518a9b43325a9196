// Centroid update: sums[f,c] += sum_{p : labels[p] == c} x_f, the three
// strategies of CentroidUpdateFactory built for gfx950:
//   cluster_merge       one LDS tile column [k*d] per work-item (no
//                       collisions), all features of the work-item's points
//                       (lloyd_cluster_merge.cl's private k x d tile)
//   feature_sum_pardim  2-D grid: blockIdx.y selects a slice of
//                       local_features*thread_features features, threadIdx.y
//                       a thread_features sub-slice; private LDS columns
//                       (lloyd_feature_sum_pardim.cl's points x feature tiles)
//   feature_sum         one LDS accumulator [d][k] shared by the work-group,
//                       work-items stride over the flattened feature-major
//                       matrix (coalesced rows)
// With every launch key at its default (names_kernel) each strategy takes the
// kernel that is fastest for the sizes (the results are the same): cluster_merge's private
// tile for a few cells, else the cell kernel below, which shares the
// accumulators of a slice of features; the strategies' own kernels serve the
// launch keys that name them.
// Every coordinate is rounded to its grid integer and added exactly
// (clk_grid.hpp): the private int32 columns flush into the work-group's
// int64 accumulator (ds_add_u64) at least every 64 values, shared
// accumulators take ds_add_u64 directly.  The work-group's sums (times the
// unit) form its FP64 partial row; the merge adds the rows (exact).  So every
// strategy and geometry gives the same bits.  The FP64 global-atomic pass (of
// grid values, so exact as well) remains for k beyond the LDS.  `masses` is
// not read, as in the reference kernels.
#include "clk_common.hpp"
#include "clk_finalize.hpp"
#include "clk_grid.hpp"
#include "clk_kernels.hpp"

#include <algorithm>
#include <type_traits>

namespace clk {
namespace {

__host__ __device__ constexpr uint32_t align4u(uint32_t v) { return (v + 3u) & ~3u; }

// LDS words before a kernel's tile: scales [nf] | acc [nf][k] int64 |
// flags [nf][k].
__host__ __device__ inline uint32_t acc_head_words(uint32_t nf, uint32_t k)
{
    return align4u(nf) + 2u * nf * k + align4u(nf * k);
}

struct AccHead {
    float *scl;
    long long *acc;
    uint32_t *flg;
    uint32_t *tail;
};

// Carve the head; stage the scales of features f0 .. f0+nf-1 and zero the
// accumulator and flags (callers add a barrier).
__device__ inline AccHead acc_head(void *lds, uint32_t nf, uint32_t k, uint32_t f0, uint32_t d,
                                   const GridRef &grid, uint32_t tid, uint32_t nthreads)
{
    AccHead h;
    h.scl = static_cast<float *>(lds);
    h.acc = reinterpret_cast<long long *>(h.scl + align4u(nf));
    h.flg = reinterpret_cast<uint32_t *>(h.acc + (size_t)nf * k);
    h.tail = h.flg + align4u(nf * k);
    for (uint32_t j = tid; j < nf; j += nthreads)
        h.scl[j] = f0 + j < d ? grid_scale(grid.gmax[f0 + j], grid.bits) : 1.0f;
    for (uint32_t i = tid; i < nf * k; i += nthreads) {
        h.acc[i] = 0;
        h.flg[i] = 0u;
    }
    return h;
}

// Add x (feature slot j of the head) of a point of cluster c into an int32
// private cell, flagging off-grid values.
__device__ __forceinline__ void add_private(uint32_t *cell, float x, float scale, const AccHead &h,
                                            uint32_t j, uint32_t k, uint32_t c)
{
    bool ok;
    const int32_t q = grid_q(x, scale, ok);
    lds_add(cell, (uint32_t)q);
    if (__builtin_expect(!ok, 0))
        lds_or(h.flg + j * k + c, special_flag(x));
}

template <int DMAX, int VEC, int BLOCK>
__global__ void __launch_bounds__(BLOCK > 0 ? BLOCK : 1024)
cu_cluster_merge_kernel(const float *__restrict__ pts, uint64_t n, uint32_t d, uint32_t k,
                        const uint32_t *__restrict__ labels, GridRef grid, double *__restrict__ part)
{
    extern __shared__ __align__(16) float lds_cm[];
    const uint32_t B = BLOCK > 0 ? BLOCK : blockDim.x;
    const uint32_t tid = threadIdx.x;
    const uint32_t rows = k * d;
    const AccHead h = acc_head(lds_cm, d, k, 0, d, grid, tid, B);
    uint32_t *tile = h.tail;  // [k*d][B] int32 grid sums
    for (uint32_t i = tid; i < rows * B; i += B)
        tile[i] = 0u;
    __syncthreads();
    uint32_t *mine = tile + tid;
    const uint32_t row_stride = d * B;
    const uint64_t groups = n / VEC;
    const uint64_t stride = (uint64_t)gridDim.x * B;
    // a cell takes at most VEC values per step: flush every 64 / VEC steps
    constexpr uint32_t kFlushSteps = 64 / VEC;
    uint32_t since = 0;
    auto flush = [&]() {
        uint32_t c = tid % k;
        for (uint32_t i = 0; i < k; ++i) {
            uint32_t *cell = mine + __umul24(c, row_stride);
#pragma unroll 1
            for (uint32_t f = 0; f < d; ++f, cell += B) {
                const int32_t v = (int32_t)*cell;
                *cell = 0u;
                lds_add64(h.acc + f * k + c, (long long)v);
            }
            c = (c + 1 == k) ? 0u : c + 1;
        }
    };
    // grid scales in registers for small buckets, read from LDS otherwise
    constexpr bool kRegScale = DMAX <= 16;
    float sc_reg[kRegScale ? DMAX : 1];
    if constexpr (kRegScale) {
#pragma unroll
        for (int f = 0; f < DMAX; ++f)
            sc_reg[f] = h.scl[f];
    }
    auto scale_of = [&](int f) -> float {
        if constexpr (kRegScale)
            return sc_reg[f];
        else
            return h.scl[f];
    };
    // the points' own grid with no NaN / inf in them: every coordinate is on
    // the grid (no range checks, no flags)
    const bool on_grid = grid.own != 0 && grid.gmax[d] == 0;
    // V points p .. p+V-1 (V = VEC, or 1 for the n % VEC tail points)
    auto add_points = [&](const auto &x, const auto &lab) {
        constexpr int V = (int)(sizeof(lab) / sizeof(uint32_t));
#pragma unroll
        for (int v = 0; v < V; ++v) {
            if (lab[v] >= k)
                continue;
            uint32_t *t = mine + __umul24(lab[v], row_stride);
            if (on_grid) {
#pragma unroll
                for (int f = 0; f < DMAX; ++f)
                    if (f < (int)d)
                        lds_add(t + f * B, (uint32_t)grid_q_on(x[f][v], scale_of(f)));
            } else {
#pragma unroll
                for (int f = 0; f < DMAX; ++f)
                    if (f < (int)d)
                        add_private(t + f * B, x[f][v], scale_of(f), h, (uint32_t)f, k, lab[v]);
            }
        }
        if (++since == kFlushSteps) {
            flush();
            since = 0;
        }
    };
    auto load = [&](uint64_t gg, float (&x)[DMAX][VEC], uint32_t (&l)[VEC]) {
        load_points<DMAX, VEC>(pts, n, d, gg * VEC, x);
        load_labels<VEC>(labels, gg * VEC, l);
    };
    uint64_t g = (uint64_t)blockIdx.x * B + tid;
    if constexpr (DMAX * VEC <= 32) {
        // Software pipeline, two register buffers: one step's points and
        // labels are in flight while the other step's are accumulated.
        // Loads are unconditional (index clamped to the last group, always
        // in bounds).  (Wider steps would not fit the registers twice.)
        const uint64_t last = groups ? groups - 1 : 0;
        float xa[DMAX][VEC], xb[DMAX][VEC];
        uint32_t la[VEC], lb[VEC];
        if (groups)
            load(min(g, last), xa, la);
        while (g < groups) {
            const uint64_t g1 = g + stride;
            load(min(g1, last), xb, lb);
            add_points(xa, la);
            if (g1 >= groups)
                break;
            const uint64_t g2 = g1 + stride;
            load(min(g2, last), xa, la);
            add_points(xb, lb);
            g = g2;
        }
    } else {
        for (; g < groups; g += stride) {
            float x[DMAX][VEC];
            uint32_t l[VEC];
            load(g, x, l);
            add_points(x, l);
        }
    }
    if constexpr (VEC > 1) {
        // the n % VEC points after the last group, one at a time, by the
        // work-item that would take group `groups` next
        if ((uint64_t)blockIdx.x * B + tid == groups % stride) {
            for (uint64_t p = groups * VEC; p < n; ++p) {
                float x1[DMAX][1];
                uint32_t l1[1];
                load_points<DMAX, 1>(pts, n, d, p, x1);
                load_labels<1>(labels, p, l1);
                add_points(x1, l1);
            }
        }
    }
    if (since != 0)
        flush();
    __syncthreads();
    for (uint32_t i = tid; i < rows; i += B) {
        const uint32_t f = i / k;  // i = f*k + c
        part[(uint64_t)blockIdx.x * rows + i] = cell_value(h.acc[i], grid_unit(h.scl[f]), h.flg[i]);
    }
}

// blockDim = (Bx, lf); block (x, y) owns features [y*FS, y*FS+FS), FS = lf*tf;
// thread (tx, ty) owns features y*FS + ty*tf + [0, tf) of points
// x*Bx + tx + i*gridDim.x*Bx.  Private LDS rows c*FS + (ty*tf + j), columns tx.
__global__ void __launch_bounds__(1024)
cu_pardim_kernel(const float *__restrict__ pts, uint64_t n, uint32_t d, uint32_t k, uint32_t tf,
                 const uint32_t *__restrict__ labels, GridRef grid, double *__restrict__ part)
{
    extern __shared__ __align__(16) float lds_pd[];
    const uint32_t Bx = blockDim.x, lf = blockDim.y;
    const uint32_t FS = lf * tf;
    const uint32_t f0 = blockIdx.y * FS;
    const uint32_t tlin = threadIdx.y * Bx + threadIdx.x;
    const uint32_t nthreads = Bx * lf;
    const uint32_t rows = k * FS;
    const AccHead h = acc_head(lds_pd, FS, k, f0, d, grid, tlin, nthreads);
    uint32_t *tile = h.tail;
    for (uint32_t i = tlin; i < rows * Bx; i += nthreads)
        tile[i] = 0u;
    __syncthreads();
    const uint32_t fsub = threadIdx.y * tf;  // first feature of this thread in the slice
    const uint64_t stride = (uint64_t)gridDim.x * Bx;
    // a cell takes at most one value per point: flush every 64 points
    uint32_t since = 0;
    auto flush = [&]() {
        for (uint32_t c = 0; c < k; ++c) {
            uint32_t *t = tile + ((uint64_t)c * FS + fsub) * Bx + threadIdx.x;
            for (uint32_t j = 0; j < tf; ++j) {
                const int32_t v = (int32_t)t[j * Bx];
                t[j * Bx] = 0u;
                lds_add64(h.acc + (fsub + j) * k + c, (long long)v);
            }
        }
    };
    for (uint64_t p = (uint64_t)blockIdx.x * Bx + threadIdx.x; p < n; p += stride) {
        const uint32_t c = labels[p];
        if (c < k) {
            uint32_t *t = tile + ((uint64_t)c * FS + fsub) * Bx + threadIdx.x;
            for (uint32_t j = 0; j < tf; ++j) {
                const uint32_t f = f0 + fsub + j;
                if (f < d)
                    add_private(t + j * Bx, pts[(uint64_t)f * n + p], h.scl[fsub + j], h, fsub + j, k, c);
            }
        }
        if (++since == 64) {
            flush();
            since = 0;
        }
    }
    if (since != 0)
        flush();
    __syncthreads();
    for (uint32_t i = tlin; i < FS * k; i += nthreads) {
        const uint32_t j = i / k, c = i % k, f = f0 + j;
        if (f < d)
            part[(uint64_t)blockIdx.x * ((uint64_t)d * k) + (uint64_t)f * k + c] =
                cell_value(h.acc[i], grid_unit(h.scl[j]), h.flg[i]);
    }
}

// Shared accumulator [d][k]; work-items stride over elements e = f*n + p.
__global__ void __launch_bounds__(1024)
cu_feature_sum_kernel(const float *__restrict__ pts, uint64_t n, uint32_t d, uint32_t k,
                      const uint32_t *__restrict__ labels, GridRef grid, double *__restrict__ part)
{
    extern __shared__ __align__(16) float lds_fs[];
    const uint32_t rows = d * k;
    const AccHead h = acc_head(lds_fs, d, k, 0, d, grid, threadIdx.x, blockDim.x);
    __syncthreads();
    const uint64_t total = n * d;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += stride) {
        const uint64_t f = e / n, p = e - f * n;
        const uint32_t c = labels[p];
        if (c < k) {
            const float x = pts[e];
            bool ok;
            const int32_t q = grid_q(x, h.scl[f], ok);
            lds_add64(h.acc + f * k + c, (long long)q);
            if (__builtin_expect(!ok, 0))
                lds_or(h.flg + f * k + c, special_flag(x));
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < rows; i += blockDim.x)
        part[(uint64_t)blockIdx.x * rows + i] = cell_value(h.acc[i], grid_unit(h.scl[i / k]), h.flg[i]);
}

// Cells of a feature slice: blockIdx.y selects features [F*blockIdx.y, +F),
// the work-group shares int64 accumulators [R][F][k] in LDS.  A wave takes 64
// consecutive points per step (lane = point: F coalesced loads and the label)
// and adds each point's grid integers into its cluster's cells with ds_add_u64
// (exact, so no ordering between lanes or waves is needed); R replicas (lane
// mod R) thin out the same-cell additions of a wave when k is small.  The
// slice's values go to the work-group's partial row, or (direct, one
// work-group per slice) are added to the sums.
// Bound by the points' bytes from a few million points on: 16M points d=64
// k=1024 648 us (6.4 TB/s; 32-bit flags, four features per slice and a quarter
// more label reads took 730), d=32 k=256 339 us (6.2 TB/s).  Against the
// kernels it replaces: 400k points d=32 k=256 168 -> 16 us (a 64-bit division
// per element), 10M d=5 k=20 78 -> 46 us (one private-tile work-group per CU).
constexpr uint32_t kCellWaves = 8;

// LDS of a cell kernel: scales [F] | cells | flag bytes.
size_t cell_lds_bytes(uint32_t F, uint64_t k, uint32_t R)
{
    return ((size_t)F * 4 + 15) / 16 * 16 + (size_t)R * F * k * 8 + (F * k + 3) / 4 * 4;
}

template <int F>
__global__ void __launch_bounds__(64 * kCellWaves)
cu_cell_kernel(const float *__restrict__ pts, uint64_t n, uint32_t d, uint32_t k, const uint32_t *__restrict__ labels,
               GridRef grid, uint32_t R, double *__restrict__ part, int direct)
{
    extern __shared__ __align__(16) char lds_cell[];
    constexpr uint32_t B = 64 * kCellWaves;
    constexpr int kRing = F >= 16 ? 2 : F >= 8 ? 4 : 8;  // steps in flight
    // the wave index as a scalar: tile indices and the loop below are then
    // wave-uniform, so the ring needs no divergent control flow
    const uint32_t tid = threadIdx.x, lane = tid % 64;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / 64));
    const uint32_t f0 = blockIdx.y * F;
    const uint32_t nf = min((uint32_t)F, d - f0), cells = F * k;
    float *scl = reinterpret_cast<float *>(lds_cell);
    long long *acc = reinterpret_cast<long long *>(lds_cell + (F * 4 + 15) / 16 * 16);
    uint32_t *flg = reinterpret_cast<uint32_t *>(acc + (size_t)R * cells);  // a byte per cell
    for (uint32_t j = tid; j < F; j += B)
        scl[j] = j < nf ? grid_scale(grid.gmax[f0 + j], grid.bits) : 1.0f;
    for (uint32_t i = tid; i < R * cells; i += B)
        acc[i] = 0;
    for (uint32_t i = tid; i < (cells + 3) / 4; i += B)
        flg[i] = 0u;
    __syncthreads();
    float sc[F];
#pragma unroll
    for (int j = 0; j < F; ++j)
        sc[j] = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(scl[j])));
    const bool on_grid = grid.own != 0 && grid.gmax[d] == 0;
    long long *const mine = acc + (size_t)(lane & (R - 1)) * cells;
    const uint64_t tiles = (n + 63) / 64;
    const uint64_t stride = (uint64_t)gridDim.x * kCellWaves;
    // Every load is unconditional and in bounds (a tile past the end reads
    // the last tile, a point past the end the last point, a feature past the
    // slice its last feature; such values are never added), so no branch
    // separates a load from its use and the later tiles' loads stay in flight.
    auto load = [&](uint64_t tile, float (&v)[F], uint32_t &L) {
        const uint64_t at = tile < tiles ? tile : tiles - 1;
        const uint64_t left = n - 1 - at * 64;
        const uint32_t off = min(lane, left < 63 ? (uint32_t)left : 63u);
        const float *base = pts + at * 64 + (uint64_t)f0 * n;
#pragma unroll
        for (int j = 0; j < F; ++j)
            v[j] = stream_load(base + (uint64_t)min((uint32_t)j, nf - 1) * n + off);
        L = (labels + at * 64)[off];  // other slices read them too: cached
    };
    auto add = [&](uint64_t tile, const float (&v)[F], uint32_t L) {
        if (tile * 64 + lane >= n || L >= k)
            return;
        if (on_grid) {
#pragma unroll
            for (int j = 0; j < F; ++j)
                if (j < (int)nf)
                    lds_add64(mine + j * k + L, (long long)grid_q_on(v[j], sc[j]));
        } else {
#pragma unroll
            for (int j = 0; j < F; ++j)
                if (j < (int)nf) {
                    bool ok;
                    const int32_t q = grid_q(v[j], sc[j], ok);
                    lds_add64(mine + j * k + L, (long long)q);
                    if (__builtin_expect(!ok, 0)) {
                        const uint32_t i = j * k + L;
                        lds_or(flg + i / 4, special_flag(v[j]) << 8 * (i % 4));
                    }
                }
        }
    };
    // this wave's tiles first + i*stride, i < count: full rounds of the ring
    // in a loop with no early exit, then the partial last round
    const uint64_t first = (uint64_t)blockIdx.x * kCellWaves + wave;
    const uint64_t count = first < tiles ? (tiles - first + stride - 1) / stride : 0;
    const uint64_t rounds = count / kRing;
    const uint32_t rest = (uint32_t)(count % kRing);
    float v[kRing][F];
    uint32_t L[kRing];
#pragma unroll
    for (int s = 0; s < kRing; ++s)
        load(first + s * stride, v[s], L[s]);
    uint64_t at = first;
    for (uint64_t r = 0; r < rounds; ++r, at += kRing * stride) {
#pragma unroll
        for (int s = 0; s < kRing; ++s) {
            const uint64_t tile = at + s * stride;  // wave-uniform, < tiles
            add(tile, v[s], L[s]);
            // refill the slot once its tile is added: its registers are free
            load(tile + kRing * stride, v[s], L[s]);
        }
    }
#pragma unroll
    for (int s = 0; s < kRing; ++s)
        if (s < (int)rest)
            add(at + s * stride, v[s], L[s]);
    __syncthreads();
    double *const row = part + (uint64_t)blockIdx.x * ((uint64_t)d * k) + (uint64_t)f0 * k;
    for (uint32_t i = tid; i < nf * k; i += B) {
        long long q = 0;
        for (uint32_t r = 0; r < R; ++r)
            q += acc[(size_t)r * cells + i];
        const double value = cell_value(q, grid_unit(scl[i / k]), (flg[i / 4] >> 8 * (i % 4)) & 7u);
        row[i] = direct ? row[i] + value : value;
    }
}

using CellKernel = void (*)(const float *, uint64_t, uint32_t, uint32_t, const uint32_t *, GridRef, uint32_t, double *, int);

struct CellPlan {
    CellKernel kern = nullptr;
    uint32_t F = 0, R = 1;
    size_t lds = 0;
};

// Points of a work-group at least: it writes F*k doubles.
uint64_t cell_points(uint64_t k) { return std::max<uint64_t>(4 * k, 64 * kCellWaves); }

// The widest slice whose cells leave a CU two work-groups (every wave slot):
// each slice reads the labels again, and loads of more features overlap.
// Else the narrowest slice that fits at all.  Narrower where the points give
// the slices less than half a work-group per CU: a few work-groups then take
// one wave's additions after another (3000 points d=64 k=300 12 -> 4.6 us, all
// in one cluster 24 -> 6.3; d=128 k=130 10.9 -> 5.8).  Replicas as far as a CU
// keeps its two work-groups and k is small enough for a wave's labels to meet.
CellPlan cell_plan(const clk_context *ctx, uint64_t d, uint64_t n, uint64_t k)
{
    CellPlan p;
    const uint32_t widest = d >= 16 ? 16 : d > 4 ? 8 : d > 2 ? 4 : (uint32_t)d;
    for (uint32_t F = widest; F >= 1 && !p.F; F /= 2)
        if (cell_lds_bytes(F, k, 1) <= ctx->lds_per_block / 2 || (F == 1 && cell_lds_bytes(1, k, 1) <= ctx->lds_per_block))
            p.F = F;
    while (p.F > 1 && div_up(d, p.F) * (n / cell_points(k)) < (uint64_t)ctx->num_cus / 2)
        p.F /= 2;
    switch (p.F) {
    case 1: p.kern = cu_cell_kernel<1>; break;
    case 2: p.kern = cu_cell_kernel<2>; break;
    case 4: p.kern = cu_cell_kernel<4>; break;
    case 8: p.kern = cu_cell_kernel<8>; break;
    case 16: p.kern = cu_cell_kernel<16>; break;
    default: return p;
    }
    while (p.R < 8 && p.R * k < 128 && cell_lds_bytes(p.F, k, 2 * p.R) <= ctx->lds_per_block / 2)
        p.R *= 2;
    p.lds = cell_lds_bytes(p.F, k, p.R);
    return p;
}

using CmKernel = void (*)(const float *, uint64_t, uint32_t, uint32_t, const uint32_t *, GridRef, double *);

// Points per work-item at most (VEC x DMAX values in registers, no spills).
constexpr int cm_vec_cap(int dmax) { return dmax >= 64 ? 1 : dmax >= 32 ? 2 : 4; }

template <int DMAX, int BLOCK>
CmKernel pick_cm_block(int vec)
{
    constexpr int cap = cm_vec_cap(DMAX);
    if constexpr (cap >= 4)
        if (vec >= 4)
            return cu_cluster_merge_kernel<DMAX, 4, BLOCK>;
    if constexpr (cap >= 2)
        if (vec >= 2)
            return cu_cluster_merge_kernel<DMAX, 2, BLOCK>;
    return cu_cluster_merge_kernel<DMAX, 1, BLOCK>;
}

template <int DMAX>
CmKernel pick_cm_vec(int vec, bool b256)
{
    return b256 ? pick_cm_block<DMAX, 256>(vec) : pick_cm_block<DMAX, 0>(vec);
}

CmKernel pick_cm(int dmax, int vec, bool b256)
{
    switch (dmax) {
    case 1: return pick_cm_vec<1>(vec, b256);
    case 2: return pick_cm_vec<2>(vec, b256);
    case 4: return pick_cm_vec<4>(vec, b256);
    case 8: return pick_cm_vec<8>(vec, b256);
    case 16: return pick_cm_vec<16>(vec, b256);
    case 32: return pick_cm_vec<32>(vec, b256);
    case 64: return pick_cm_vec<64>(vec, b256);
    default: return nullptr;
    }
}

const char *const kCellNames[] = {"CentroidUpdateFeatureSum", "CentroidUpdateFeatureSumPardim",
                                  "CentroidUpdateClusterMerge"};

// Whether cluster_merge's private tile beats the shared cells: only on the
// largest data, with two work-groups per CU and enough cells (2^27 points,
// d=4 k=10: 421 us against 433; k=16: 439 / 459; but d=4 k=3 540 / 433, d=2
// k=10 277 / 261, and 16M points d=4 k=10 60 / 55).
bool private_pays(const clk_context *ctx, uint64_t n, uint64_t dk, uint64_t lds)
{
    return n >= (64u << 20) && dk >= 32 && 2 * lds <= ctx->lds_per_block;
}

}  // namespace

int run_centroid_update(clk_context *ctx, const clk_kernel_config *cfg, uint64_t d, uint64_t n,
                        uint64_t k, const float *points, double *sums, const uint32_t *labels,
                        hipStream_t stream)
{
    CLK_REQUIRE(d >= 1 && k >= 1 && k <= 0xFFFFFFFFull && d <= 0xFFFFull, CLK_ERR_SIZE,
                "centroid_update: bad d or k");
    CLK_REQUIRE(points && sums && labels, CLK_ERR_INVALID_ARGUMENT, "centroid_update: null buffer");
    if (n == 0)
        return CLK_OK;
    const int strategy = cfg ? cfg->strategy : CLK_CENTROID_CLUSTER_MERGE;
    CLK_REQUIRE(strategy >= CLK_CENTROID_FEATURE_SUM && strategy <= CLK_CENTROID_CLUSTER_MERGE,
                CLK_ERR_INVALID_ARGUMENT, "centroid_update: unknown strategy id");
    const uint64_t B = (cfg && cfg->local_size[0]) ? cfg->local_size[0] : 256;
    CLK_REQUIRE(B <= (uint64_t)ctx->max_threads_per_block, CLK_ERR_INVALID_ARGUMENT,
                "centroid_update: local_size exceeds the device limit");
    const uint64_t user_grid = (cfg && cfg->global_size[0]) ? div_up(cfg->global_size[0], B) : 0;
    const uint64_t dk = d * k;
    const int dmax = dmax_bucket(d);

    GridRef sg;
    CLK_TRY(resolve_grid(ctx, d, n, points, stream, &sg));
    const uint64_t head = (uint64_t)acc_head_words((uint32_t)d, (uint32_t)k) * 4;

    const void *kern = nullptr;
    const char *name = nullptr;
    size_t lds = 0;
    dim3 grid, block;
    uint32_t tf = 1;
    uint64_t gx = 0;

    const bool automatic = !names_kernel(cfg);
    const bool private_fits = dmax && dk < (1ull << 24) && head + dk * B * 4 <= ctx->lds_per_block;
    const CellPlan cells = cell_plan(ctx, d, n, k);
    const bool take_cells = cells.kern && automatic && !(private_fits && private_pays(ctx, n, dk, head + dk * B * 4));
    if (!take_cells && private_fits && (automatic || strategy == CLK_CENTROID_CLUSTER_MERGE)) {
        const int vec = std::min(pick_vector_width(cfg ? cfg->vector_length : 4), cm_vec_cap(dmax));
        CmKernel kc = pick_cm(dmax, vec, B == 256);
        lds = head + dk * B * 4;
        gx = user_grid ? user_grid : auto_grid(ctx, (const void *)kc, (int)B, lds, n / vec);
        gx = std::max<uint64_t>(1, std::min<uint64_t>(gx, 1u << 20));
        if (lds > 65536)
            CLK_HIP_CHECK(hipFuncSetAttribute((const void *)kc, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        CLK_TRY(ensure_scratch(ctx->part_sums, gx * dk * sizeof(double)));
        double *ps = static_cast<double *>(ctx->part_sums.ptr);
        {
            KernelTimer t(ctx, "CentroidUpdateClusterMerge", stream);
            hipLaunchKernelGGL(kc, dim3((unsigned)gx), dim3((unsigned)B), lds, stream, points, n,
                               (uint32_t)d, (uint32_t)k, labels, sg, ps);
            CLK_HIP_CHECK(hipGetLastError());
        }
        return launch_merge_sums(ctx, ps, gx, dk, sums, stream);
    }
    if (!take_cells && strategy == CLK_CENTROID_FEATURE_SUM_PARDIM) {
        uint64_t lf = (cfg && cfg->local_features) ? cfg->local_features : 1;
        tf = (uint32_t)((cfg && cfg->thread_features) ? cfg->thread_features : 1);
        lf = std::min<uint64_t>(lf, d);
        uint64_t bx = std::max<uint64_t>(1, B / lf);
        uint64_t fs = lf * tf;
        lds = (uint64_t)acc_head_words((uint32_t)fs, (uint32_t)k) * 4 + k * fs * bx * 4;
        if (k * fs < (1ull << 24) && lds <= ctx->lds_per_block && bx * lf <= (uint64_t)ctx->max_threads_per_block) {
            kern = (const void *)cu_pardim_kernel;
            block = dim3((unsigned)bx, (unsigned)lf);
            uint64_t gy = div_up(d, fs);
            gx = user_grid ? user_grid : auto_grid(ctx, kern, (int)(bx * lf), lds, n);
            gx = std::max<uint64_t>(1, std::min<uint64_t>(div_up(gx, gy), 1u << 20));
            grid = dim3((unsigned)gx, (unsigned)gy);
            name = "CentroidUpdateFeatureSumPardim";
        }
    }
    if (!kern && !take_cells && dk < (1ull << 24) && head <= ctx->lds_per_block) {
        kern = (const void *)cu_feature_sum_kernel;
        lds = head;
        block = dim3((unsigned)B);
        gx = user_grid ? user_grid : auto_grid(ctx, kern, (int)B, lds, n * d);
        gx = std::max<uint64_t>(1, std::min<uint64_t>(gx, 1u << 20));
        grid = dim3((unsigned)gx);
        name = "CentroidUpdateFeatureSum";
    }
    if (!kern && cells.kern) {
        if (cells.lds > 65536)
            CLK_HIP_CHECK(hipFuncSetAttribute((const void *)cells.kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                              (int)cells.lds));
        // A resident grid over the slices; a work-group takes at least
        // cell_points, up to 16k points where one per CU is enough (each writes
        // F*k doubles, which the merge reads: 400k points d=32 k=256 26 -> 21
        // us, 50k d=128 k=130 17.6 -> 14.5).
        const uint64_t gy = div_up(d, (uint64_t)cells.F);
        uint64_t gxs = auto_grid(ctx, (const void *)cells.kern, 64 * kCellWaves, cells.lds, n * gy) / gy;
        uint64_t share = cell_points(k);
        while (gy * div_up(n, share) > (uint64_t)ctx->num_cus && share < 16 * k)
            share *= 2;
        gxs = std::min<uint64_t>(gxs, div_up(n, share));
        gxs = std::max<uint64_t>(1, std::min<uint64_t>(gxs, 65535));
        // Few points: one work-group per slice, which adds its sums itself.
        // Its waves take the points one after another, so it pays up to about
        // what the merge's launch costs: 8192 points d=4 k=10 33.6 us a step
        // through the separate operators against 35.8, 16k d=8 k=30 even.
        const bool direct = n * cells.F <= 32768 && n <= 16384;
        // (the global atomics need no scratch memory)
        if (direct)
            gxs = 1;
        else if (!try_scratch(ctx->part_sums, gxs * dk * sizeof(double), stream))
            return launch_accumulate_global(ctx, d, n, k, points, labels, sg, sums, nullptr, stream);
        double *ps = direct ? sums : static_cast<double *>(ctx->part_sums.ptr);
        {
            KernelTimer t(ctx, kCellNames[strategy], stream);
            hipLaunchKernelGGL(cells.kern, dim3((unsigned)gxs, (unsigned)gy), dim3(64 * kCellWaves), cells.lds,
                               stream, points, n, (uint32_t)d, (uint32_t)k, labels, sg, cells.R, ps, direct);
            CLK_HIP_CHECK(hipGetLastError());
        }
        if (direct)
            return CLK_OK;
        return launch_merge_sums(ctx, ps, gxs, dk, sums, stream);
    }
    if (!kern)
        return launch_accumulate_global(ctx, d, n, k, points, labels, sg, sums, nullptr, stream);

    if (lds > 65536)
        CLK_HIP_CHECK(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    CLK_TRY(ensure_scratch(ctx->part_sums, gx * dk * sizeof(double)));
    double *ps = static_cast<double *>(ctx->part_sums.ptr);
    {
        KernelTimer t(ctx, name, stream);
        if (kern == (const void *)cu_pardim_kernel)
            hipLaunchKernelGGL(cu_pardim_kernel, grid, block, lds, stream, points, n, (uint32_t)d,
                               (uint32_t)k, tf, labels, sg, ps);
        else
            hipLaunchKernelGGL(cu_feature_sum_kernel, grid, block, lds, stream, points, n,
                               (uint32_t)d, (uint32_t)k, labels, sg, ps);
        CLK_HIP_CHECK(hipGetLastError());
    }
    return launch_merge_sums(ctx, ps, gx, dk, sums, stream);
}

}  // namespace clk

extern "C" int clk_centroid_update(clk_context *ctx, const clk_kernel_config *cfg, uint64_t d,
                                   uint64_t n, uint64_t k, const float *points, double *sums,
                                   const uint32_t *labels, const uint32_t *masses, void *stream)
{
    (void)masses;
    CLK_TRY(clk::enter(ctx));
    CLK_REQUIRE(!cfg || cfg->stage == CLK_STAGE_CENTROID_UPDATE, CLK_ERR_INVALID_ARGUMENT,
                "clk_centroid_update: config is not a centroid-update-stage config");
    return clk::run_centroid_update(ctx, cfg, d, n, k, points, sums, labels,
                                    clk::as_stream(stream));
}
