// Labeling pass and fused pass with split-operand MFMA labels (clk_split.hpp)
// for the sizes where the sequential-fma scan is bound by its vector
// operations: 2 per feature and centroid plus the argmin, against 2.5 per
// centroid for ranking matrix-core scores.  Measured with the launches
// included, before -> now: fused step 2.5M points d=7 k=33 71 -> 44 us (13 of
// them the points' bytes), 700k d=24 k=48 113 -> 45; 2^20 d=4 k=10 21.5 -> 18;
// labeling 400k d=32 k=256 183 -> 44 us.  What is left is issue-bound: about
// 150 vector instructions per 64 points and 60 per tile of 16 centroids, the
// matrix core (64 cycles per tile at P <= 8) only partly under them.
#include "clk_common.hpp"
#include "clk_finalize.hpp"
#include "clk_grid.hpp"
#include "clk_kernels.hpp"
#include "clk_split.hpp"

#include <algorithm>

namespace clk {
namespace {

using namespace split;

// Waves per work-group: one per SIMD where the operands need more than 256
// registers.
constexpr uint32_t split_waves(int P) { return P >= 96 ? 4 : 8; }

// LDS words after the table of a fused pass: scales [P] | acc [R][d*k] int64
// | flags [d*k] | counts [R][k].  R replicas (lane mod R) thin out the
// same-cell atomics of a wave.
__host__ __device__ inline size_t fused_tail_bytes(uint32_t P, uint32_t d, uint32_t k, uint32_t R)
{
    return (size_t)P * 4 + (size_t)R * d * k * 8 + (size_t)d * k * 4 + (size_t)R * k * 4 + 16;
}

// FUSED: labels, masses and grid-exact sums (clk_grid.hpp) in one pass, the
// work-group's partial row to part (clk_finalize.hpp); else labels only.
// A wave takes 64 consecutive points per step.  P <= 16: lane = point, the
// next step's coordinates loaded while this step is labelled.  P >= 32: lane
// (q, h) holds features 8h .. 8h+7 of each K-block of the points q, 16+q,
// 32+q, 48+q (the matrix core's layout).
template <int P, bool FUSED>
__global__ void __launch_bounds__(64 * split_waves(P))
split_kernel(const float *__restrict__ pts, uint64_t n, uint32_t d, uint32_t k, const float *__restrict__ cen,
             uint32_t *__restrict__ labels, uint32_t ntiles, GridRef grid, uint32_t R, double *__restrict__ part,
             double *__restrict__ max_shift)
{
    using Sh = Shape<P>;
    constexpr uint32_t kWaves = split_waves(P);
    extern __shared__ __align__(16) char smem_split[];
    const uint32_t tid = threadIdx.x, lane = tid % 64, B = 64 * kWaves;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / 64));
    const uint32_t q = lane % 16, h = lane / 16;
    const uint32_t dk = d * k;
    // the exchange planes end the table's block; the fused tail follows
    u16x8 *buf = reinterpret_cast<u16x8 *>(smem_split + lds_bytes<P>(ntiles, 0)) + wave * Sh::planes * 64;
    char *tail = smem_split + lds_bytes<P>(ntiles, kWaves);
    float *scl = reinterpret_cast<float *>(tail);
    long long *acc = reinterpret_cast<long long *>(scl + P);
    uint32_t *flg = reinterpret_cast<uint32_t *>(acc + (size_t)R * dk);
    uint32_t *cnt = flg + dk;
    if constexpr (FUSED) {
        if (max_shift && blockIdx.x == 0 && tid == 0)
            *max_shift = 0.0;  // the merge raises it
        for (uint32_t f = tid; f < P; f += B)
            scl[f] = f < d ? grid_scale(grid.gmax[f], grid.bits) : 1.0f;
        for (uint32_t i = tid; i < R * dk; i += B)
            acc[i] = 0;
        for (uint32_t i = tid; i < dk; i += B)
            flg[i] = 0u;
        for (uint32_t i = tid; i < R * k; i += B)
            cnt[i] = 0u;
    }
    const Table t = stage<P>(cen, d, k, ntiles, smem_split);
    const bool on_grid = FUSED && grid.own != 0 && grid.gmax[d] == 0;

    constexpr int kOwn = P < 32 ? P : Sh::nkb * 8;  // coordinates per lane and point
    constexpr int kPts = P < 32 ? 1 : 4;            // points a lane holds parts of
    float sc[FUSED ? kOwn : 1];
    if constexpr (FUSED) {
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            sc[i] = scl[P < 32 ? i : (i / 8) * 32 + 8 * h + i % 8];
            if constexpr (P < 32)  // wave-uniform: a scalar register
                sc[i] = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(sc[i])));
        }
    }
    auto feature = [&](int i) -> uint32_t { return P < 32 ? (uint32_t)i : (uint32_t)(i / 8) * 32 + 8 * h + i % 8; };

    // Every load is unconditional and in bounds: a point past the end reads
    // point n-1, a feature past d reads feature d-1 (0 in the centroids, never
    // added), so no branch stands between the loads and the next step's stay
    // in flight.
    uint32_t rows[P < 32 ? 1 : kOwn];  // P >= 32: this lane's row offsets
    if constexpr (P >= 32)
#pragma unroll
        for (int i = 0; i < kOwn; ++i)
            rows[i] = min(feature(i), d - 1) * (uint32_t)n;  // n * d <= 2^30
    auto load = [&](uint64_t bt, float (&x)[kPts][kOwn]) {
        const float *base = pts + bt * 64;                              // wave-uniform
        const uint64_t left = n - 1 - bt * 64;
        const uint32_t last = left < 63 ? (uint32_t)left : 63u;
#pragma unroll
        for (int g = 0; g < kPts; ++g) {
            const uint32_t off = min(P < 32 ? lane : g * 16 + q, last);
#pragma unroll
            for (int i = 0; i < kOwn; ++i) {
                if constexpr (P < 32)
                    x[g][i] = stream_load(base + (uint64_t)min((uint32_t)i, d - 1) * n + off);
                else
                    x[g][i] = base[rows[i] + off];
            }
        }
    };
    auto step = [&](uint64_t bt, const float (&x)[kPts][kOwn]) {
        const uint64_t p = bt * 64 + lane;
        PointOps<P> ops;
        float x2, best, second;
        if constexpr (P < 32)
            x2 = build_points<P>(x[0], t.scale, buf, lane, ops);
        else
            x2 = build_points<P>(x, t.scale, lane, ops);
        rank_points<P>(t, ops, lane, best, second);
        uint32_t lab;
        const bool sure = decide(t, x2, best, second, k, lab);
        uint64_t open = __ballot(!sure && p < n);
        if constexpr (P < 32) {
            // Many undecided points against few centroids: every lane scans
            // for its own point (about k (2P + 3) instructions in all, against
            // about 150 for each point that the wave scans together).
            if (open && k * (2 * P + 3) <= 150u * (uint32_t)__builtin_popcountll(open)) {
                float own[P][1];
#pragma unroll
                for (int f = 0; f < P; ++f)
                    own[f][0] = f < (int)d ? x[0][f] : 0.0f;
                uint32_t scanned[1];
                argmin_lds<P, 1>(own, t.rows, k, scanned);
                lab = sure ? lab : scanned[0];
                open = 0;
            }
        }
        if (open)
            exact_scan(open, pts + bt * 64, n, cen, d, k, lane, lab);
        if (p < n)
            stream_store(lab, labels + p);
        if constexpr (FUSED) {
            long long *const mine = acc + (size_t)(lane & (R - 1)) * dk;
            if (p < n)
                lds_add(cnt + (lane & (R - 1)) * k + lab, 1u);
#pragma unroll
            for (int g = 0; g < kPts; ++g) {
                const uint32_t lg = P < 32 ? lab : (uint32_t)__shfl((int)lab, (int)(g * 16 + q));
                const bool in = bt * 64 + (P < 32 ? lane : g * 16 + q) < n;
                if (on_grid) {
                    if (in) {
#pragma unroll
                        for (int i = 0; i < kOwn; ++i)
                            if (feature(i) < d)
                                lds_add64(mine + feature(i) * k + lg, (long long)grid_q_on(x[g][i], sc[i]));
                    }
                } else if (in) {
#pragma unroll
                    for (int i = 0; i < kOwn; ++i)
                        if (feature(i) < d) {
                            bool ok;
                            const int32_t v = grid_q(x[g][i], sc[i], ok);
                            lds_add64(mine + feature(i) * k + lg, (long long)v);
                            if (!ok)  // added as 0, its cell flagged
                                lds_or(flg + feature(i) * k + lg, special_flag(x[g][i]));
                        }
                }
            }
        }
    };
    const uint64_t batches = (n + 63) / 64;
    const uint64_t stride = (uint64_t)gridDim.x * kWaves;
    uint64_t bt = (uint64_t)blockIdx.x * kWaves + wave;
    if constexpr (P <= 32) {
        // two register buffers: the next step's loads are in flight
        float xa[kPts][kOwn], xb[kPts][kOwn];
        load(bt < batches ? bt : batches - 1, xa);
        while (bt < batches) {
            const uint64_t b1 = bt + stride;
            load(b1 < batches ? b1 : batches - 1, xb);
            step(bt, xa);
            if (b1 >= batches)
                break;
            bt = b1 + stride;
            load(bt < batches ? bt : batches - 1, xa);
            step(b1, xb);
        }
    } else {
        for (; bt < batches; bt += stride) {
            float x[kPts][kOwn];
            load(bt, x);
            step(bt, x);
        }
    }
    if constexpr (FUSED) {
        __syncthreads();
        double *const row = part + (uint64_t)blockIdx.x * (dk + k);
        for (uint32_t i = tid; i < dk; i += B) {
            long long s = 0;
            for (uint32_t r = 0; r < R; ++r)
                s += acc[(size_t)r * dk + i];
            row[i] = cell_value(s, grid_unit(scl[i / k]), flg[i]);
        }
        for (uint32_t c = tid; c < k; c += B) {
            uint32_t s = 0;
            for (uint32_t r = 0; r < R; ++r)
                s += cnt[r * k + c];
            row[dk + c] = (double)s;
        }
    }
}

using SplitKernel = void (*)(const float *, uint64_t, uint32_t, uint32_t, const float *, uint32_t *, uint32_t, GridRef,
                             uint32_t, double *, double *);

struct SplitPlan {
    SplitKernel kern = nullptr;
    uint32_t block = 0;
    uint32_t ntiles = 0, R = 1;
    size_t lds = 0;
};

template <int P, bool FUSED>
SplitPlan plan_for(const clk_context *ctx, uint64_t d, uint64_t k)
{
    SplitPlan p;
    p.ntiles = (uint32_t)div_up(k, (uint64_t)16);
    p.block = 64 * split_waves(P);
    p.lds = lds_bytes<P>(p.ntiles, split_waves(P));
    if (FUSED) {
        // replicas only where they leave the CU its second work-group
        p.R = P < 32 ? 4 : 1;
        while (p.R > 1 && p.lds + fused_tail_bytes(P, (uint32_t)d, (uint32_t)k, p.R) > ctx->lds_per_block / 2)
            p.R /= 2;
        p.lds += fused_tail_bytes(P, (uint32_t)d, (uint32_t)k, p.R);
    }
    if (p.lds <= ctx->lds_per_block)
        p.kern = split_kernel<P, FUSED>;
    return p;
}

template <bool FUSED>
SplitPlan split_plan(const clk_context *ctx, uint64_t d, uint64_t k)
{
    if (d == 0 || k == 0 || k > 65536)
        return {};
    if (d <= 4)
        return plan_for<4, FUSED>(ctx, d, k);
    if (d <= 8)
        return plan_for<8, FUSED>(ctx, d, k);
    if (d <= 16)
        return plan_for<16, FUSED>(ctx, d, k);
    if (d <= 32)
        return plan_for<32, FUSED>(ctx, d, k);
    if constexpr (!FUSED) {
        if (d <= 64)
            return plan_for<64, FUSED>(ctx, d, k);
        if (d <= 96)
            return plan_for<96, FUSED>(ctx, d, k);
        if (d <= 128)
            return plan_for<128, FUSED>(ctx, d, k);
    }
    return {};
}

uint64_t split_grid(clk_context *ctx, const SplitPlan &p, uint64_t n)
{
    return auto_grid(ctx, (const void *)p.kern, (int)p.block, p.lds, n);
}

int allow_lds(const SplitPlan &p)
{
    if (p.lds > 65536)
        CLK_HIP_CHECK(hipFuncSetAttribute((const void *)p.kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds));
    return CLK_OK;
}

}  // namespace

bool split_labeling_pays(const clk_context *ctx, const clk_kernel_config *cfg, uint64_t d, uint64_t n, uint64_t k,
                         bool fused)
{
    // an explicit launch geometry names the plain kernels' one
    if (cfg && (cfg->global_size[0] || (cfg->local_size[0] && cfg->local_size[0] != 256)))
        return false;
    if (d > 16 && n * d > (1ull << 30))  // 32-bit row offsets
        return false;
    // Where the line lies (us, this pass against the plain kernels, 2M points
    // unless said).  Labeling: d=4 k=20 18.3 / 13.7, k=32 17.6 / 18.7; d=8
    // k=16 17.8 / 20.8; d=16 k=16 31 / 39; d=32 k=10 60 / 55, k=16 55 / 65;
    // with one or two features the plain scan's 2d + 3 operations per centroid
    // stay below the ranking's.  Fused step: d=4 k=3 33 / 34, k=10 25 / 29,
    // k=50 36 / 47; d=16 k=5 61 / 50, k=10 52 / 73; d=32 k=32 88 / 190; 300k
    // points d=4 k=5 14 / 19, d=16 k=3 22 / 35; 20k points d=4 k=5 11 / 16.
    // One feature and many clusters: the gaps sink below the keys' truncation
    // (274k points k=238: 81 / 45) and the plain scan costs 5 per centroid.
    if (fused)
        return (k >= 6 || (n <= (1u << 20) && k >= 2)) && (d > 1 || k <= 32) &&
               split_plan<true>(ctx, d, k).kern != nullptr;
    const uint64_t bucket = d <= 4 ? 4 : d <= 8 ? 8 : d <= 16 ? 16 : div_up(d, (uint64_t)32) * 32;
    return n >= 4096 && d >= 3 && k * (2 * bucket + 3) >= 300 + 20 * bucket &&
           split_plan<false>(ctx, d, k).kern != nullptr;
}

int launch_labeling_split(clk_context *ctx, const char *name, uint64_t d, uint64_t n, uint64_t k, const float *points,
                          const float *centroids, uint32_t *labels, hipStream_t stream)
{
    const SplitPlan p = split_plan<false>(ctx, d, k);
    CLK_REQUIRE(p.kern && n > 0, CLK_ERR_UNSUPPORTED, "split labeling: sizes");
    CLK_TRY(allow_lds(p));
    KernelTimer t(ctx, name, stream);
    hipLaunchKernelGGL(p.kern, dim3((unsigned)split_grid(ctx, p, n)), dim3(p.block), p.lds, stream, points, n,
                       (uint32_t)d, (uint32_t)k, centroids, labels, p.ntiles, GridRef{}, 1u,
                       nullptr, nullptr);
    CLK_HIP_CHECK(hipGetLastError());
    return CLK_OK;
}

uint64_t fused_split_rows(clk_context *ctx, uint64_t d, uint64_t n, uint64_t k)
{
    return split_grid(ctx, split_plan<true>(ctx, d, k), n);
}

int launch_fused_split(clk_context *ctx, const char *name, uint64_t d, uint64_t n, uint64_t k, const float *points,
                       const float *centroids, uint32_t *labels, const GridRef &grid, uint64_t rows, double *part,
                       double *max_shift, hipStream_t stream)
{
    const SplitPlan p = split_plan<true>(ctx, d, k);
    CLK_REQUIRE(p.kern && n > 0, CLK_ERR_UNSUPPORTED, "split fused pass: sizes");
    CLK_TRY(allow_lds(p));
    KernelTimer t(ctx, name, stream);
    hipLaunchKernelGGL(p.kern, dim3((unsigned)rows), dim3(p.block), p.lds, stream, points, n, (uint32_t)d,
                       (uint32_t)k, centroids, labels, p.ntiles, grid, p.R, part, max_shift);
    CLK_HIP_CHECK(hipGetLastError());
    return CLK_OK;
}

}  // namespace clk
