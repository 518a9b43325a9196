// Labeling pass and fused pass with split-operand MFMA labels (clk_split.hpp)
// for the sizes where the sequential-fma scan is bound by its vector
// operations: 2 per feature and centroid plus the argmin, against 2.5 per
// centroid for ranking matrix-core scores.  Measured with the launches
// included, before -> now: fused step 2.5M points d=7 k=33 71 -> 45 us (13 of
// them the points' bytes), 700k d=24 k=48 113 -> 45, 5M double d=4 k=10 58 ->
// 53; labeling 400k d=32 k=256 187 -> 53 us.  What is left is issue-bound: about
// 150 vector instructions per 64 points and 60 per tile of 16 centroids, the
// matrix core (64 cycles per tile at P <= 8) only partly under them.
#include "clk_common.hpp"
#include "clk_finalize.hpp"
#include "clk_grid.hpp"
#include "clk_kernels.hpp"
#include "clk_split.hpp"

#include <algorithm>
#include <type_traits>

namespace clk {
namespace {

using namespace split;

// Waves per work-group: one per SIMD where the operands need more than 256
// registers.
constexpr uint32_t split_waves(int P) { return P >= 96 ? 4 : 8; }

// Waves per SIMD that the registers have to leave room for: two work-groups to
// a CU up to 8 features, and of the four-wave ones at 96 (float points).
constexpr uint32_t split_occupancy(int P, bool f64) { return P <= 8 ? 4 : P <= 64 || (P == 96 && !f64) ? 2 : 1; }

// LDS after the table of a fused pass: scales [P] | cells [R][d*k] | flags
// [d*k] | counts [R][k].  Float points: int64 cells of grid integers
// (clk_grid.hpp); double points: FP64 cells, no scales or flags.  R replicas
// (lane mod R) thin out the same-cell atomics of a wave.
__host__ __device__ inline size_t fused_tail_bytes(uint32_t P, uint32_t d, uint32_t k, uint32_t R, bool f64)
{
    return (f64 ? 0 : (size_t)P * 4 + (size_t)d * k * 4) + (size_t)R * d * k * 8 + (size_t)R * k * 4 + 16;
}

// FUSED: labels, masses and sums in one pass, the work-group's partial row to
// part (clk_finalize.hpp); else labels only.
// A wave takes 64 consecutive points per step.  P <= 16: lane = point, the
// next step's coordinates loaded while this step is labelled.  P >= 32: lane
// (q, h) holds features 8h .. 8h+7 of each K-block of the points q, 16+q,
// 32+q, 48+q (the matrix core's layout).
template <int P, bool FUSED, typename T, typename LabelT>
__global__ void __launch_bounds__(64 * split_waves(P), split_occupancy(P, sizeof(T) == 8))
split_kernel(const T *__restrict__ pts, uint64_t n, uint32_t d, uint32_t k, const T *__restrict__ cen,
             LabelT *__restrict__ labels, uint32_t ntiles, GridRef grid, uint32_t R, double *__restrict__ part,
             double *__restrict__ max_shift)
{
    using Sh = Shape<P>;
    constexpr bool f64 = sizeof(T) == 8;
    using Cell = std::conditional_t<f64, double, long long>;
    constexpr uint32_t kWaves = split_waves(P);
    extern __shared__ __align__(16) char smem_split[];
    const uint32_t tid = threadIdx.x, lane = tid % 64, B = 64 * kWaves;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / 64));
    const uint32_t q = lane % 16, h = lane / 16;
    const uint32_t dk = d * k;
    // the exchange planes end the table's block; the fused tail follows
    u16x8 *buf = reinterpret_cast<u16x8 *>(smem_split + lds_bytes<P, T>(ntiles, 0)) + wave * Sh::planes * 64;
    char *tail = smem_split + lds_bytes<P, T>(ntiles, kWaves);
    float *scl = reinterpret_cast<float *>(tail);
    Cell *acc = reinterpret_cast<Cell *>(scl + (f64 ? 0 : P));
    uint32_t *flg = reinterpret_cast<uint32_t *>(acc + (size_t)R * dk);
    uint32_t *cnt = flg + (f64 ? 0 : dk);
    if constexpr (FUSED) {
        if (max_shift && blockIdx.x == 0 && tid == 0)
            *max_shift = 0.0;  // the merge raises it
        for (uint32_t i = tid; i < R * dk; i += B)
            acc[i] = 0;
        if constexpr (!f64) {
            for (uint32_t f = tid; f < P; f += B)
                scl[f] = f < d ? grid_scale(grid.gmax[f], grid.bits) : 1.0f;
            for (uint32_t i = tid; i < dk; i += B)
                flg[i] = 0u;
        }
        for (uint32_t i = tid; i < R * k; i += B)
            cnt[i] = 0u;
    }
    const Table<T> t = stage<P, T>(cen, d, k, ntiles, smem_split);
    const bool on_grid = FUSED && !f64 && grid.own != 0 && grid.gmax[d] == 0;

    constexpr int kOwn = P < 32 ? P : Sh::nkb * 8;  // coordinates per lane and point
    constexpr int kPts = P < 32 ? 1 : 4;            // points a lane holds parts of
    constexpr bool kScales = FUSED && !f64;
    float sc[kScales ? kOwn : 1];
    if constexpr (kScales) {
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
    auto load = [&](uint64_t bt, T (&x)[kPts][kOwn]) {
        const T *base = pts + bt * 64;                              // wave-uniform
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
    auto step = [&](uint64_t bt, const T (&x)[kPts][kOwn]) {
        const uint64_t p = bt * 64 + lane;
        PointOps<P> ops;
        float x2, best, second;
        if constexpr (P < 32)
            x2 = build_points<P, T>(t, x[0], buf, lane, ops);
        else
            x2 = build_points<P, T>(t, x, lane, ops);
        rank_points<P, T>(t, ops, lane, best, second);
        uint32_t lab;
        float limit;
        const bool sure = decide(t, x2, best, second, k, lab, limit);
        uint64_t open = __ballot(!sure && p < n);  // points that the wave scans one by one
        const uint32_t m = (uint32_t)__builtin_popcountll(open), rounds = (k + 63) / 64;
        bool all = false;  // every lane scans for its own point, and the ones that are not sure take that
        if constexpr (P < 32) {
            // about k (2P + 3) instructions, against about 150 for each point
            // and 64 centroids that the wave scans together (double points: the
            // rows take twice the LDS reads; 150k points d=8 k=700 172 / 243 us
            // without that)
            all = open && k * (2 * P + 3) <= 150u * m * (f64 ? (rounds + 1) / 2 : rounds);
        } else if (open) {
            all = m > 5;  // (block_scan)
            if constexpr (!(f64 && !FUSED && P == 32)) {  // (its registers spill)
                // Scoring the tiles again and one exact distance a lane for each
                // tile with candidates, against the rounds of the full scan:
                // 188k points d=53 k=290 with clusters sharing blobs 640 ->
                // 203 us.
                const uint64_t known = __ballot(!sure && p < n && limit == limit);
                const uint32_t mk = (uint32_t)__builtin_popcountll(known);
                const uint32_t full = k > 32 ? mk * rounds : k > 16 ? (mk + 1) / 2 : (mk + 3) / 4;
                if (m - mk <= 5 && full > min(ntiles, 2 * mk) + ntiles / 8 + 1)
                    if (candidate_scan<P>(t, ops, known, limit, pts + bt * 64, n, cen, d, k, lane, lab)) {
                        open &= ~known;
                        all = false;
                    }
            }
        }
        if (all) {
            uint32_t scanned;
            if constexpr (P < 32) {
                scanned = scan_rows<P, T>(t, x[0], d, k);
            } else {
                const uint64_t left = n - 1 - bt * 64;
                const T *own = pts + bt * 64 + min(lane, left < 63 ? (uint32_t)left : 63u);
                scanned = block_scan(own, n, cen, d, k, lane);
            }
            lab = sure ? lab : scanned;
        } else if (open) {
            exact_scan<P>(open, pts + bt * 64, n, cen, d, k, lane, lab);
        }
        if (p < n)
            stream_store((LabelT)lab, labels + p);
        if constexpr (FUSED) {
            Cell *const mine = acc + (size_t)(lane & (R - 1)) * dk;
            if (p < n)
                lds_add(cnt + (lane & (R - 1)) * k + lab, 1u);
#pragma unroll
            for (int g = 0; g < kPts; ++g) {
                const uint32_t lg = P < 32 ? lab : (uint32_t)__shfl((int)lab, (int)(g * 16 + q));
                const bool in = bt * 64 + (P < 32 ? lane : g * 16 + q) < n;
                if constexpr (f64) {
                    if (in) {
#pragma unroll
                        for (int i = 0; i < kOwn; ++i)
                            if (feature(i) < d)
                                atomicAdd(mine + feature(i) * k + lg, x[g][i]);
                    }
                } else if (on_grid) {
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
    if constexpr (P <= 32 && !(f64 && FUSED && P == 32)) {
        // two register buffers: the next step's loads are in flight
        T xa[kPts][kOwn], xb[kPts][kOwn];
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
            T x[kPts][kOwn];
            load(bt, x);
            step(bt, x);
        }
    }
    if constexpr (FUSED) {
        __syncthreads();
        double *const row = part + (uint64_t)blockIdx.x * (dk + k);
        for (uint32_t i = tid; i < dk; i += B) {
            Cell s = 0;
            for (uint32_t r = 0; r < R; ++r)
                s += acc[(size_t)r * dk + i];
            if constexpr (f64)
                row[i] = s;
            else
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

template <typename T>
using LabelOf = std::conditional_t<sizeof(T) == 8, uint64_t, uint32_t>;
template <typename T>
using SplitKernel = void (*)(const T *, uint64_t, uint32_t, uint32_t, const T *, LabelOf<T> *, uint32_t, GridRef, uint32_t,
                             double *, double *);

template <typename T>
struct SplitPlan {
    SplitKernel<T> kern = nullptr;
    uint32_t block = 0;
    uint32_t ntiles = 0, R = 1;
    size_t lds = 0;
};

template <int P, bool FUSED, typename T>
SplitPlan<T> plan_for(const clk_context *ctx, uint64_t d, uint64_t k)
{
    constexpr bool f64 = sizeof(T) == 8;
    SplitPlan<T> p;
    p.ntiles = (uint32_t)div_up(k, (uint64_t)16);
    p.block = 64 * split_waves(P);
    p.lds = lds_bytes<P, T>(p.ntiles, split_waves(P));
    if (FUSED) {
        // replicas only where they leave the CU its second work-group
        p.R = P < 32 ? 4 : 1;
        while (p.R > 1 && p.lds + fused_tail_bytes(P, (uint32_t)d, (uint32_t)k, p.R, f64) > ctx->lds_per_block / 2)
            p.R /= 2;
        p.lds += fused_tail_bytes(P, (uint32_t)d, (uint32_t)k, p.R, f64);
    }
    if (p.lds <= ctx->lds_per_block)
        p.kern = split_kernel<P, FUSED, T, LabelOf<T>>;
    return p;
}

template <bool FUSED, typename T>
SplitPlan<T> split_plan(const clk_context *ctx, uint64_t d, uint64_t k)
{
    if (d == 0 || k < 2 || k > 65536)
        return {};
    if (d <= 4)
        return plan_for<4, FUSED, T>(ctx, d, k);
    if (d <= 8)
        return plan_for<8, FUSED, T>(ctx, d, k);
    if (d <= 16)
        return plan_for<16, FUSED, T>(ctx, d, k);
    if (d <= 32)
        return plan_for<32, FUSED, T>(ctx, d, k);
    if constexpr (!FUSED) {
        if (d <= 64)
            return plan_for<64, FUSED, T>(ctx, d, k);
        if (d <= 96)
            return plan_for<96, FUSED, T>(ctx, d, k);
        if (d <= 128)
            return plan_for<128, FUSED, T>(ctx, d, k);
    }
    return {};
}

// Padded features of the plans.
uint64_t split_bucket(uint64_t d)
{
    return d <= 4 ? 4 : d <= 8 ? 8 : d <= 16 ? 16 : div_up(d, (uint64_t)32) * 32;
}

template <typename T>
uint64_t split_grid(clk_context *ctx, const SplitPlan<T> &p, uint64_t n)
{
    return auto_grid(ctx, (const void *)p.kern, (int)p.block, p.lds, n);
}

template <typename T>
int launch_split(clk_context *ctx, const SplitPlan<T> &p, const char *name, uint64_t grid, uint64_t d, uint64_t n,
                 uint64_t k, const T *points, const T *centroids, LabelOf<T> *labels, const GridRef &sgrid,
                 double *part, double *max_shift, hipStream_t stream)
{
    CLK_REQUIRE(p.kern && n > 0, CLK_ERR_UNSUPPORTED, "split labels: sizes");
    if (p.lds > 65536)
        CLK_HIP_CHECK(hipFuncSetAttribute((const void *)p.kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds));
    KernelTimer t(ctx, name, stream);
    hipLaunchKernelGGL(p.kern, dim3((unsigned)grid), dim3(p.block), p.lds, stream, points, n, (uint32_t)d, (uint32_t)k,
                       centroids, labels, p.ntiles, sgrid, p.R, part, max_shift);
    CLK_HIP_CHECK(hipGetLastError());
    return CLK_OK;
}

}  // namespace

bool split_labeling_pays(const clk_context *ctx, const clk_kernel_config *cfg, uint64_t d, uint64_t n, uint64_t k,
                         bool fused)
{
    if (names_kernel(cfg))
        return false;
    if (d > 16 && n * d > (1ull << 30))  // 32-bit row offsets
        return false;
    // Where the line lies (us, this pass against the plain kernels, 2M points
    // unless said).  Labeling: d=4 k=20 18.3 / 13.7, k=32 17.6 / 18.7; d=8
    // k=16 17.8 / 20.8; d=16 k=16 31 / 39; d=32 k=10 60 / 55, k=16 55 / 65;
    // with one or two features the plain scan's 2d + 3 operations per centroid
    // stay below the ranking's.  Fused step: d=16 k=5 61 / 50, k=10 52 / 73;
    // d=32 k=32 88 / 190; 300k points d=16 k=3 22 / 35, but two clusters of more
    // than 16 features 400k d=32 75 / 54, 1M d=20 57 / 48.
    // One feature: the gaps sink below the keys' truncation (2M points k=8 20 /
    // 11, k=20 26 / 12, 274k k=238 81 / 45); the plain scan takes 5 operations
    // a centroid.
    // Up to four features the plain pass (shared cells) is the faster one
    // until the scan is long: 3M points d=4 k=10 26.0 / 25.1, k=24 30.8 / 30.5,
    // k=48 36 / 45; 300k d=4 k=24 12.3 / 9.9, k=48 12.8 / 12.6; d=3 k=32 11.9 /
    // 10.6, k=48 12.8 / 12.2, 3M 36 / 41; d=2 k=150 3M 79 / 67.
    if (fused && d <= 4)
        return d >= 3 && k >= 48 && split_plan<true, float>(ctx, d, k).kern != nullptr;
    if (fused)
        return (k >= 6 || (n <= (1u << 20) && k >= (d > 16 ? 3u : 2u))) &&
               split_plan<true, float>(ctx, d, k).kern != nullptr;
    const uint64_t bucket = split_bucket(d);
    return n >= 4096 && d >= 3 && k * (2 * bucket + 3) >= 300 + 20 * bucket &&
           split_plan<false, float>(ctx, d, k).kern != nullptr;
}

int launch_labeling_split(clk_context *ctx, const char *name, uint64_t d, uint64_t n, uint64_t k, const float *points,
                          const float *centroids, uint32_t *labels, hipStream_t stream)
{
    const SplitPlan<float> p = split_plan<false, float>(ctx, d, k);
    return launch_split(ctx, p, name, p.kern ? split_grid(ctx, p, n) : 0, d, n, k, points, centroids, labels, GridRef{},
                        nullptr, nullptr, stream);
}

uint64_t fused_split_rows(clk_context *ctx, uint64_t d, uint64_t n, uint64_t k)
{
    return split_grid(ctx, split_plan<true, float>(ctx, d, k), n);
}

int launch_fused_split(clk_context *ctx, const char *name, uint64_t d, uint64_t n, uint64_t k, const float *points,
                       const float *centroids, uint32_t *labels, const GridRef &grid, uint64_t rows, double *part,
                       double *max_shift, hipStream_t stream)
{
    return launch_split(ctx, split_plan<true, float>(ctx, d, k), name, rows, d, n, k, points, centroids, labels, grid,
                        part, max_shift, stream);
}

// ---- double points ---------------------------------------------------------

uint64_t split_rows_f64(clk_context *ctx, const clk_kernel_config *cfg, uint64_t d, uint64_t n, uint64_t k, bool fused)
{
    if (cfg && (cfg->global_size[0] || (cfg->local_size[0] && cfg->local_size[0] != 256)))
        return 0;
    if (n == 0 || (d > 16 && n * d > (1ull << 30)))
        return 0;
    // Where the line lies (us, this pass against f64_pass_kernel).  Labeling:
    // 2M points d=4 k=16 19 / 22, k=8 18 / 18; d=8 k=16 29 / 39; d=32 k=8 120 /
    // 120, k=100 151 / 576; 200k d=8 k=32 8.5 / 12; 20k d=8 k=32 6.8 / 7.7, d=4
    // k=100 10 / 8.  Fused step: 2M d=4 k=4 32 / 37; d=2 k=32 31 / 38, k=8 24 /
    // 23; d=32 k=32 139 / 299; 200k d=8 k=4 16 / 17, d=4 k=16 15 / 15; 20k d=8
    // k=32 12 / 13, k=16 12 / 10.  One feature: the plain scan always.
    const uint64_t b = split_bucket(d), cost = k * (2 * b + 3);
    bool pays;
    if (d <= 2)
        pays = fused && d == 2 && n >= 1000000 && k >= 32;
    else if (n >= 1000000)
        pays = fused || cost >= 150 + 10 * b;
    else if (n >= 100000)
        pays = fused ? b >= 8 || cost >= 300 : cost >= 300 + 20 * b;
    else
        pays = b >= 8 && cost >= 600;
    if (!pays)
        return 0;
    const SplitPlan<double> p = fused ? split_plan<true, double>(ctx, d, k) : split_plan<false, double>(ctx, d, k);
    return p.kern && k >= 2 ? split_grid(ctx, p, n) : 0;
}

int launch_split_f64(clk_context *ctx, const char *name, uint64_t d, uint64_t n, uint64_t k, const double *points,
                     const double *centroids, uint64_t *labels, uint64_t rows, double *part, double *max_shift,
                     hipStream_t stream)
{
    const SplitPlan<double> p = part ? split_plan<true, double>(ctx, d, k) : split_plan<false, double>(ctx, d, k);
    return launch_split(ctx, p, name, rows, d, n, k, points, centroids, labels, GridRef{}, part, max_shift, stream);
}

}  // namespace clk
