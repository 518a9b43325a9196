// The sum grid (clk_grid.hpp): per-feature max |x| pass, the context's
// pinned grid and its C ABI.
#include "clk_grid.hpp"
#include "clk_kernels.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

namespace clk {
namespace {

constexpr int kGridBlock = 1024;

// The maximum of n values of a row over the work-items t0, t0 + stride, ...
// (four 128-bit loads in flight each; NaN and +-inf are skipped), into *gmax:
// bits of non-negative floats order like their values; NaN or +-inf set
// *special_seen.  At most one atomicMax per work-group: device atomics on one
// address take about 45 ns each.
__device__ __forceinline__ void grid_max_row(const float *__restrict__ row, uint64_t n, uint64_t t0, uint64_t stride,
                                             uint32_t *__restrict__ gmax, uint32_t *__restrict__ special_seen)
{
    __shared__ uint32_t wave_max[kGridBlock / kWave];
    uint32_t m = 0;
    bool special = false;  // a NaN or an infinity seen
    auto take = [&](float x) {
        const float a = __builtin_fabsf(x);
        const uint32_t u = __float_as_uint(a);
        const bool fin = a <= FLT_MAX;
        m = (fin && u > m) ? u : m;
        special = special || !fin;
    };
    auto take4 = [&](const gf32x4 &v) {
        take(v.x);
        take(v.y);
        take(v.z);
        take(v.w);
    };
    // 128-bit loads (4-byte aligned rows), then the n % 4 tail values
    const gf32x4 *r4 = reinterpret_cast<const gf32x4 *>(row);
    const uint64_t n4 = n / 4;
    uint64_t i = t0;
    for (; i + 3 * stride < n4; i += 4 * stride) {
        gf32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            v[u] = stream_load(r4 + i + u * stride);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            take4(v[u]);
    }
    for (; i < n4; i += stride)
        take4(stream_load(r4 + i));
    if (t0 < n % 4)
        take(row[n4 * 4 + t0]);
    for (int o = 32; o >= 1; o /= 2) {
        const uint32_t other = (uint32_t)__shfl_xor((int)m, o);
        m = other > m ? other : m;
    }
    // a finite maximum never has the sign bit: it carries the special flag
    const bool any = __ballot(special) != 0;
    if (threadIdx.x % kWave == 0)
        wave_max[threadIdx.x / kWave] = m | (any ? 0x80000000u : 0u);
    __syncthreads();
    if (threadIdx.x != 0)
        return;
    uint32_t best = 0, flags = 0;
    for (int w = 0; w < kGridBlock / kWave; ++w) {
        const uint32_t u = wave_max[w] & 0x7FFFFFFFu;
        best = u > best ? u : best;
        flags |= wave_max[w];
    }
    // plain look first: most work-groups have nothing to raise
    if (best > __hip_atomic_load(gmax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(gmax, best);
    if ((flags & 0x80000000u) && !__hip_atomic_load(special_seen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicOr(special_seen, 1u);
}

// blockIdx.y = feature; the work-items of blockIdx.x stride over the row.  With
// one atomic per work-group (one per wave bounded the pass), launch included,
// before -> now: 2^20 points d=4 51 -> 14 us; 2.5M d=7 60 -> 29; 10M d=5
// 81 -> 45; 2^27 d=4 382 -> 320 (6.7 TB/s).
__global__ void __launch_bounds__(kGridBlock)
grid_max_kernel(const float *__restrict__ pts, uint64_t n, uint32_t *__restrict__ gmax, uint32_t d)
{
    const uint32_t f = blockIdx.y;
    grid_max_row(pts + (uint64_t)f * n, n, (uint64_t)blockIdx.x * kGridBlock + threadIdx.x,
                 (uint64_t)gridDim.x * kGridBlock, gmax + f, gmax + d);
}

// Slices of rows of several point sets (cleared gmax), one per work-group.
__global__ void __launch_bounds__(kGridBlock) grid_max_units_kernel(const GridUnit *__restrict__ units)
{
    const GridUnit u = units[blockIdx.x];
    grid_max_row(u.values, u.count, threadIdx.x, kGridBlock, u.gmax, u.special_seen);
}

}  // namespace

int launch_grid_max(clk_context *ctx, uint64_t d, uint64_t n, const float *points, uint32_t *gmax,
                    hipStream_t stream)
{
    CLK_TRY(clk_fill_zero(ctx, gmax, (d + 1) * sizeof(uint32_t), stream));
    if (n == 0)
        return CLK_OK;
    CLK_REQUIRE(d <= 65535, CLK_ERR_SIZE, "sum grid: d too large");
    // two work-groups per CU over all features (every wave slot), at least
    // one 128-bit load per work-item, at most 256 atomics per feature
    const uint64_t per_row = std::min<uint64_t>(256, div_up(2 * (uint64_t)ctx->num_cus, d));
    const uint64_t gx = std::min<uint64_t>(per_row, div_up(n, kGridBlock * 4));
    KernelTimer t(ctx, "SumGrid", stream);
    hipLaunchKernelGGL(grid_max_kernel, dim3((unsigned)std::max<uint64_t>(gx, 1), (unsigned)d),
                       dim3(kGridBlock), 0, stream, points, n, gmax, (uint32_t)d);
    CLK_HIP_CHECK(hipGetLastError());
    return CLK_OK;
}

int launch_grid_max_units(clk_context *ctx, const GridUnit *units, uint32_t count, hipStream_t stream)
{
    KernelTimer t(ctx, "SumGrid", stream);
    hipLaunchKernelGGL(grid_max_units_kernel, dim3(count), dim3(kGridBlock), 0, stream, units);
    CLK_HIP_CHECK(hipGetLastError());
    return CLK_OK;
}

int resolve_grid(clk_context *ctx, uint64_t d, uint64_t n, const float *points, hipStream_t stream,
                 GridRef *out)
{
    if (ctx->grid_pinned) {
        CLK_REQUIRE(ctx->grid_d == d, CLK_ERR_INVALID_ARGUMENT,
                    "the sum grid pinned on the context has another number of features");
        out->gmax = static_cast<const uint32_t *>(ctx->grid.ptr);
        out->bits = grid_bits(ctx->grid_n);
        out->own = ctx->grid_src != nullptr && ctx->grid_src == points && ctx->grid_n == n;
        return CLK_OK;
    }
    CLK_TRY(ensure_scratch(ctx->grid, (d + 1) * sizeof(uint32_t)));
    CLK_TRY(launch_grid_max(ctx, d, n, points, static_cast<uint32_t *>(ctx->grid.ptr), stream));
    out->gmax = static_cast<const uint32_t *>(ctx->grid.ptr);
    out->bits = grid_bits(n);
    out->own = 1;
    return CLK_OK;
}

}  // namespace clk

using namespace clk;

extern "C" int clk_sum_grid_from_points(clk_context *ctx, uint64_t d, uint64_t n, const float *points,
                                        void *stream)
{
    CLK_TRY(enter(ctx));
    CLK_REQUIRE(d >= 1 && d <= 65535, CLK_ERR_SIZE, "clk_sum_grid_from_points: bad d");
    CLK_REQUIRE(points || n == 0, CLK_ERR_INVALID_ARGUMENT, "clk_sum_grid_from_points: null points");
    ctx->grid_pinned = false;
    CLK_TRY(ensure_scratch(ctx->grid, (d + 1) * sizeof(uint32_t)));
    CLK_TRY(launch_grid_max(ctx, d, n, points, static_cast<uint32_t *>(ctx->grid.ptr), as_stream(stream)));
    ctx->grid_pinned = true;
    ctx->grid_d = d;
    ctx->grid_n = n;
    ctx->grid_src = points;
    return CLK_OK;
}

extern "C" int clk_sum_grid_from_max(clk_context *ctx, uint64_t d, uint64_t n, const float *host_max_abs)
{
    CLK_TRY(enter(ctx));
    CLK_REQUIRE(d >= 1 && d <= 65535, CLK_ERR_SIZE, "clk_sum_grid_from_max: bad d");
    CLK_REQUIRE(host_max_abs != nullptr, CLK_ERR_INVALID_ARGUMENT, "clk_sum_grid_from_max: null maxima");
    std::vector<uint32_t> bits(d + 1, 0u);
    for (uint64_t f = 0; f < d; ++f) {
        const float a = std::fabs(host_max_abs[f]);
        uint32_t u = 0;
        if (a <= FLT_MAX)
            std::memcpy(&u, &a, 4);
        bits[f] = u;
    }
    bits[d] = 1u;  // whether the data hold NaN / inf is not known: check
    ctx->grid_pinned = false;
    CLK_TRY(ensure_scratch(ctx->grid, (d + 1) * sizeof(uint32_t)));
    CLK_HIP_CHECK(hipMemcpy(ctx->grid.ptr, bits.data(), (d + 1) * sizeof(uint32_t), hipMemcpyHostToDevice));
    ctx->grid_pinned = true;
    ctx->grid_d = d;
    ctx->grid_n = n;
    ctx->grid_src = nullptr;
    return CLK_OK;
}

extern "C" int clk_sum_grid_clear(clk_context *ctx)
{
    CLK_REQUIRE(ctx != nullptr, CLK_ERR_INVALID_ARGUMENT, "null clk_context");
    ctx->grid_pinned = false;
    ctx->grid_src = nullptr;
    return CLK_OK;
}

extern "C" int clk_sum_grid_units(clk_context *ctx, uint64_t d, uint64_t n, const float *points,
                                  double *host_units, void *stream)
{
    CLK_TRY(enter(ctx));
    CLK_REQUIRE(host_units != nullptr, CLK_ERR_INVALID_ARGUMENT, "clk_sum_grid_units: null output");
    CLK_REQUIRE(d >= 1 && d <= 65535, CLK_ERR_SIZE, "clk_sum_grid_units: bad d");
    hipStream_t s = as_stream(stream);
    GridRef g;
    CLK_TRY(resolve_grid(ctx, d, n, points, s, &g));
    std::vector<uint32_t> bits(d);
    CLK_HIP_CHECK(hipMemcpyAsync(bits.data(), g.gmax, d * sizeof(uint32_t), hipMemcpyDeviceToHost, s));
    CLK_HIP_CHECK(hipStreamSynchronize(s));
    for (uint64_t f = 0; f < d; ++f)
        host_units[f] = grid_unit(grid_scale(bits[f], g.bits));
    return CLK_OK;
}
