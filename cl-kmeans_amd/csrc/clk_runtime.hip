// Context, error reporting, per-kernel timing, and the small element-wise /
// reduction kernels of the Lloyd iteration: fill, first_x, matrix add,
// column-vector reduction (ReduceVectorParcol) and the FP64 divide
// (MatrixBinaryOp::row).
#include "clk_common.hpp"
#include "clk_finalize.hpp"
#include "clk_kernels.hpp"

#include <algorithm>
#include <cstring>
#include <mutex>

namespace clk {

static thread_local std::string g_last_error;

void set_error(const std::string &msg) { g_last_error = msg; }

int enter(clk_context *ctx)
{
    CLK_REQUIRE(ctx != nullptr, CLK_ERR_INVALID_ARGUMENT, "null clk_context");
    CLK_HIP_CHECK(hipSetDevice(ctx->device));
    return CLK_OK;
}

int ensure_scratch(Scratch &s, size_t bytes)
{
    if (s.bytes >= bytes)
        return CLK_OK;
    if (s.ptr) {
        CLK_HIP_CHECK(hipFree(s.ptr));
        s.ptr = nullptr;
        s.bytes = 0;
    }
    size_t want = std::max<size_t>(bytes, 4096);
    hipError_t e = hipMalloc(&s.ptr, want);
    if (e != hipSuccess) {
        s.ptr = nullptr;
        set_error(std::string("scratch hipMalloc failed: ") + hipGetErrorString(e));
        return CLK_ERR_NOMEM;
    }
    s.bytes = want;
    return CLK_OK;
}

bool try_scratch(Scratch &s, size_t bytes, hipStream_t stream)
{
    if (s.bytes >= bytes)
        return true;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    const bool free_stream = hipStreamIsCapturing(stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone;
    const bool grown = free_stream && ensure_scratch(s, bytes) == CLK_OK;
    if (!grown)
        (void)hipGetLastError();
    return grown;
}

static hipEvent_t take_event(clk_context *ctx)
{
    if (!ctx->event_pool.empty()) {
        hipEvent_t e = ctx->event_pool.back();
        ctx->event_pool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess)
        return nullptr;
    return e;
}

KernelTimer::KernelTimer(clk_context *c, const char *name, hipStream_t s) : ctx(c), stream(s)
{
    if (!ctx->profiling)
        return;
    hipEvent_t a = take_event(ctx), b = take_event(ctx);
    if (!a || !b)
        return;
    ctx->records.push_back(TimingRecord{name, ctx->iteration, a, b});
    rec = (int64_t)ctx->records.size() - 1;
    (void)hipEventRecord(a, stream);
}

KernelTimer::~KernelTimer()
{
    if (rec >= 0)
        (void)hipEventRecord(ctx->records[(size_t)rec].stop, stream);
}

int pick_vector_width(uint64_t requested)
{
    if (requested == 1 || requested == 2 || requested == 4)
        return (int)requested;
    return 4;
}

uint64_t auto_grid(clk_context *ctx, const void *kernel, int block, size_t dyn_lds,
                   uint64_t work_items)
{
    int per_cu = 0;
    for (const clk_context::Occupancy &o : ctx->occupancies)
        if (o.kernel == kernel && o.block == block && o.lds == dyn_lds)
            per_cu = o.per_cu;
    if (per_cu == 0) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, dyn_lds) !=
                hipSuccess ||
            per_cu < 1)
            per_cu = 1;
        if (ctx->occupancies.size() >= 64)  // sizes that keep changing
            ctx->occupancies.clear();
        ctx->occupancies.push_back({kernel, block, per_cu, dyn_lds});
    }
    uint64_t grid = (uint64_t)per_cu * (uint64_t)ctx->num_cus;
    uint64_t need = div_up(std::max<uint64_t>(work_items, 1), (uint64_t)block);
    return std::max<uint64_t>(1, std::min(grid, need));
}

// ------------------------------------------------------------ kernels ---

namespace {

__global__ void fill_zero_kernel(uint4 *__restrict__ p16, uint64_t n16,
                                 uint8_t *__restrict__ tail, uint64_t ntail)
{
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t j = i; j < n16; j += stride)
        p16[j] = make_uint4(0, 0, 0, 0);
    for (uint64_t j = i; j < ntail; j += stride)
        tail[j] = 0;
}

__global__ void first_x_kernel(const float *__restrict__ pts, uint64_t n, uint32_t d,
                               uint32_t k, float *__restrict__ cen)
{
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (uint64_t)d * k)
        return;
    uint64_t f = i / k, c = i % k;
    cen[i] = pts[f * n + (c % n)];
}

template <typename T>
__global__ void matrix_add_kernel(T *__restrict__ fst, const T *__restrict__ snd, uint64_t count)
{
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (; i < count; i += stride)
        fst[i] = fst[i] + snd[i];
}

// Column reduction with a fixed order.  A block covers 64 rows with
// G = blockDim.x/64 column groups; thread (lane, g) sums columns
// g, g+G, g+2G, ... of row r0+lane into four interleaved accumulators
// (independent load chains), combines them as (a0+a1)+(a2+a3), and the G
// group sums are added in group order.  `in` and `out` may alias (in-place):
// a block reads and writes only its own rows.
template <typename T>
__device__ __forceinline__ T column_sum(const T *in, uint64_t cols, uint64_t rows, uint64_t r,
                                        uint32_t g, uint32_t G)
{
    T a0 = 0, a1 = 0, a2 = 0, a3 = 0;
    uint64_t c = g;
    for (; c + 3 * (uint64_t)G < cols; c += 4 * (uint64_t)G) {
        a0 += in[c * rows + r];
        a1 += in[(c + G) * rows + r];
        a2 += in[(c + 2 * (uint64_t)G) * rows + r];
        a3 += in[(c + 3 * (uint64_t)G) * rows + r];
    }
    for (; c < cols; c += G)
        a0 += in[c * rows + r];
    return (T)((T)(a0 + a1) + (T)(a2 + a3));
}

template <typename T>
__global__ void __launch_bounds__(1024) reduce_cols_kernel(const T *in, uint64_t cols,
                                                           uint64_t rows, T *out)
{
    __shared__ T part[1024];
    const uint32_t lane = threadIdx.x % 64, g = threadIdx.x / 64;
    const uint32_t G = blockDim.x / 64;
    const uint64_t r = (uint64_t)blockIdx.x * 64 + lane;
    part[threadIdx.x] = (r < rows) ? column_sum(in, cols, rows, r, g, G) : (T)0;
    __syncthreads();
    if (g == 0 && r < rows) {
        T t = part[lane];
        for (uint32_t j = 1; j < G; ++j)
            t += part[j * 64 + lane];
        out[r] = t;
    }
}

// centroids[f,c] = (float)(sums[f,c] / (double)masses[c]) without a shift: a
// work-item per value (one work-group over all of them, below, takes 26 us at
// d=64 k=1024).
__global__ void __launch_bounds__(256) divide_values_kernel(const double *__restrict__ sums,
                                                            const uint32_t *__restrict__ masses, uint32_t count,
                                                            uint32_t k, float *__restrict__ cen)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < count)
        cen[i] = (float)(sums[i] / (double)masses[i % k]);
}

// centroids[f,c] = (float)(sums[f,c] / (double)masses[c]); optional max
// centroid shift (FP64) over non-empty clusters.  One block.
__global__ void __launch_bounds__(1024) divide_kernel(const double *__restrict__ sums,
                                                      const uint32_t *__restrict__ masses,
                                                      uint32_t d, uint32_t k,
                                                      float *__restrict__ cen,
                                                      const float *__restrict__ old_cen,
                                                      double *__restrict__ max_shift)
{
    __shared__ double red[1024];
    double local_max = 0.0;
    for (uint32_t c = threadIdx.x; c < k; c += blockDim.x) {
        const double m = (double)masses[c];
        double sq = 0.0;
        for (uint32_t f = 0; f < d; ++f) {
            const uint64_t i = (uint64_t)f * k + c;
            const float v = (float)(sums[i] / m);
            cen[i] = v;
            if (old_cen) {
                const double diff = (double)v - (double)old_cen[i];
                sq += diff * diff;
            }
        }
        if (masses[c] != 0u)
            local_max = fmax(local_max, sqrt(sq));
    }
    if (!max_shift || !old_cen)
        return;
    red[threadIdx.x] = local_max;
    __syncthreads();
    for (uint32_t s = blockDim.x / 2; s > 0; s /= 2) {
        if (threadIdx.x < s)
            red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0)
        *max_shift = red[0];
}

}  // namespace

// 64 rows x up to 16 column groups; fewer groups for few columns.
static unsigned reduce_block(uint64_t cols)
{
    unsigned groups = 1;
    while (groups < 16 && (uint64_t)groups * 8 < cols)
        groups *= 2;
    return 64 * groups;
}

namespace {

constexpr uint32_t kMergeThreads = 1024;

// A work-group merges `clusters` clusters of every value row: lane j of the
// a.lanes value lanes holds value row j / clusters of cluster
// blockIdx.x * clusters + j % clusters, and the kMergeThreads / lanes row
// groups stride over the partial rows with eight loads in flight each, so a
// thread waits for memory about rows / (8 * groups) times; the groups' sums
// meet in LDS.  The work is latency first, then the rows' bytes.  One
// work-group over all values (the form this replaces) against this kernel,
// launch included: d=4 k=10, 768 rows 12.9 -> 8.1 us; d=7 k=33, 2048 rows
// 64 -> 21 us; d=24 k=48, 1536 rows 152 -> 35 us.
template <typename In, typename MassT, typename CenT>
__global__ void __launch_bounds__(kMergeThreads) merge_kernel(MergeArgs<In, MassT, CenT> a)
{
    __shared__ In part[kMergeThreads];
    __shared__ double diff[kMergeThreads];
    const uint32_t tid = threadIdx.x, L = a.lanes, G = kMergeThreads / L;
    const uint32_t j = tid % L, g = tid / L;
    const uint32_t nv = a.d + (a.mass ? 1u : 0u), C = a.clusters;
    const uint32_t f = j / C, jc = j % C;
    const uint64_t c = (uint64_t)blockIdx.x * C + jc;
    const bool active = f < nv && c < a.k;
    const uint64_t row = nv * a.k;  // values of a partial row
    In acc[8] = {};
    if (active) {
        const In *p = a.part + f * a.k + c;
        uint32_t r = g;
        for (; r + 7 * G < a.rows; r += 8 * G) {
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u)
                acc[u] += p[(uint64_t)(r + u * G) * row];
        }
        // the last up to seven rows: clamped loads, so they too are issued
        // together
        if (r < a.rows) {
#pragma unroll
            for (uint32_t u = 0; u < 7; ++u) {
                const uint32_t q = r + u * G;
                const In v = p[(uint64_t)min(q, a.rows - 1) * row];
                acc[u] += q < a.rows ? v : (In)0;
            }
        }
    }
    part[tid] = (In)(((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7])));
    __syncthreads();
    for (uint32_t s = G / 2; s > 0; s /= 2) {
        if (g < s)
            part[tid] += part[tid + s * L];
        __syncthreads();
    }
    const In t = part[j];
    if (g == 0 && active) {
        const uint64_t i = f * a.k + c;
        if (f >= a.d) {
            a.masses[c] = a.divide ? (MassT)t : (MassT)(a.masses[c] + (MassT)t);
        } else if (!a.divide) {
            a.sums[i] += (double)t;
        } else {
            // FP64 divide, one rounding to CenT; an empty cluster gives 0/0 = NaN
            a.sums[i] = (double)t;
            const CenT v = (CenT)((double)t / (double)part[a.d * C + jc]);
            a.centroids[i] = v;
            if (a.max_shift)
                diff[j] = (double)v - (double)a.old_centroids[i];
        }
    }
    if (!a.divide || !a.max_shift)
        return;
    __syncthreads();
    if (tid < C && c < a.k && part[a.d * C + j] != (In)0) {
        double sq = 0.0;
        for (uint32_t q = 0; q < a.d; ++q)
            sq += diff[q * C + j] * diff[q * C + j];
        // a NaN move (old centroid NaN) does not count; non-negative doubles
        // order like their bit patterns; the plain load spares most of the
        // same-address atomics
        const unsigned long long u = (unsigned long long)__double_as_longlong(fmax(0.0, sqrt(sq)));
        unsigned long long *const m = reinterpret_cast<unsigned long long *>(a.max_shift);
        if (u > __hip_atomic_load(m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(m, u);
    }
}

}  // namespace

template <typename In, typename MassT, typename CenT>
int launch_merge(clk_context *ctx, MergeArgs<In, MassT, CenT> a, const char *name, hipStream_t stream)
{
    const uint32_t nv = a.d + (a.mass ? 1u : 0u);
    if (nv == 0 || a.k == 0 || a.rows == 0)
        return CLK_OK;
    CLK_REQUIRE(nv <= kMergeThreads, CLK_ERR_SIZE, "merge: too many value rows");
    // At most eight rows per thread where 16 value lanes allow it; as many
    // value lanes as that leaves, at least one per value row.
    uint32_t lanes = 16;
    while (lanes < 256 && (uint64_t)(kMergeThreads / lanes) * 4 >= a.rows)
        lanes *= 2;
    while (lanes < nv)
        lanes *= 2;
    a.lanes = lanes;
    a.clusters = (uint32_t)std::min<uint64_t>(lanes / nv, a.k);
    KernelTimer t(ctx, name, stream);
    hipLaunchKernelGGL((merge_kernel<In, MassT, CenT>), dim3((unsigned)div_up(a.k, a.clusters)),
                       dim3(kMergeThreads), 0, stream, a);
    CLK_HIP_CHECK(hipGetLastError());
    return CLK_OK;
}

template int launch_merge(clk_context *, MergeF32, const char *, hipStream_t);
template int launch_merge(clk_context *, MergeF64, const char *, hipStream_t);
template int launch_merge(clk_context *, MergeU32, const char *, hipStream_t);

int launch_reduce_f64(clk_context *ctx, const double *in, uint64_t cols, uint64_t rows,
                      double *out, hipStream_t stream)
{
    if (rows == 0)
        return CLK_OK;
    KernelTimer t(ctx, "ReduceVectorParcol", stream);
    hipLaunchKernelGGL(reduce_cols_kernel<double>, dim3((unsigned)div_up(rows, 64)),
                       dim3(reduce_block(cols)), 0, stream, in, cols, rows, out);
    CLK_HIP_CHECK(hipGetLastError());
    return CLK_OK;
}

int launch_reduce_u32(clk_context *ctx, const uint32_t *in, uint64_t cols, uint64_t rows,
                      uint32_t *out, hipStream_t stream)
{
    if (rows == 0)
        return CLK_OK;
    KernelTimer t(ctx, "ReduceVectorParcol", stream);
    hipLaunchKernelGGL(reduce_cols_kernel<uint32_t>, dim3((unsigned)div_up(rows, 64)),
                       dim3(reduce_block(cols)), 0, stream, in, cols, rows, out);
    CLK_HIP_CHECK(hipGetLastError());
    return CLK_OK;
}

}  // namespace clk

using namespace clk;

// -------------------------------------------------------------- C ABI ---

extern "C" const char *clk_last_error(void) { return g_last_error.c_str(); }

// For the host layer's C entry points (C++ exceptions -> clk_last_error).
extern "C" void clk_set_error_message(const char *msg) { clk::set_error(msg ? msg : ""); }

extern "C" int clk_context_create(int device, clk_context **out)
{
    CLK_REQUIRE(out != nullptr, CLK_ERR_INVALID_ARGUMENT, "clk_context_create: null out");
    *out = nullptr;
    int count = 0;
    CLK_HIP_CHECK(hipGetDeviceCount(&count));
    CLK_REQUIRE(device >= 0 && device < count, CLK_ERR_INVALID_ARGUMENT,
                "clk_context_create: no such HIP device");
    CLK_HIP_CHECK(hipSetDevice(device));
    hipDeviceProp_t prop;
    CLK_HIP_CHECK(hipGetDeviceProperties(&prop, device));
    clk_context *ctx = new clk_context;
    ctx->device = device;
    ctx->num_cus = prop.multiProcessorCount;
    ctx->lds_per_block = prop.sharedMemPerBlock;
    ctx->max_threads_per_block = prop.maxThreadsPerBlock;
    const int rc = noalloc_setup(ctx);
    if (rc != CLK_OK) {
        delete ctx;
        return rc;
    }
    *out = ctx;
    return CLK_OK;
}

extern "C" int clk_context_destroy(clk_context *ctx)
{
    if (!ctx)
        return CLK_OK;
    (void)hipSetDevice(ctx->device);
    (void)hipDeviceSynchronize();
    if (ctx->part_sums.ptr)
        (void)hipFree(ctx->part_sums.ptr);
    for (clk::Scratch *sc : {&ctx->part_masses, &ctx->mfma_tables, &ctx->mfma_queue, &ctx->mfma_hint, &ctx->mfma_pin, &ctx->grid})
        if (sc->ptr)
            (void)hipFree(sc->ptr);
    for (auto &r : ctx->records) {
        (void)hipEventDestroy(r.start);
        (void)hipEventDestroy(r.stop);
    }
    for (auto e : ctx->event_pool)
        (void)hipEventDestroy(e);
    delete ctx;
    return CLK_OK;
}

extern "C" int clk_strategy_id(int stage, const char *name)
{
    CLK_REQUIRE(name != nullptr, CLK_ERR_INVALID_ARGUMENT, "clk_strategy_id: null name");
    std::string s(name);
    switch (stage) {
    case CLK_STAGE_FUSED:
        if (s == "cluster_merge") return CLK_FUSED_CLUSTER_MERGE;
        if (s == "feature_sum") return CLK_FUSED_FEATURE_SUM;
        if (s == "cluster_merge_bounded") return CLK_FUSED_CLUSTER_MERGE_BOUNDED;
        break;
    case CLK_STAGE_LABELING:
        if (s == "unroll_vector") return CLK_LABELING_UNROLL_VECTOR;
        if (s == "mfma_bf16") return CLK_LABELING_MFMA_BF16;
        if (s == "mfma_fp16") return CLK_LABELING_MFMA_FP16;
        if (s == "unroll_vector_bounded") return CLK_LABELING_UNROLL_VECTOR_BOUNDED;
        break;
    case CLK_STAGE_MASS_UPDATE:
        if (s == "global_atomic") return CLK_MASS_GLOBAL_ATOMIC;
        if (s == "part_global") return CLK_MASS_PART_GLOBAL;
        if (s == "part_local") return CLK_MASS_PART_LOCAL;
        if (s == "part_private") return CLK_MASS_PART_PRIVATE;
        break;
    case CLK_STAGE_CENTROID_UPDATE:
        if (s == "feature_sum") return CLK_CENTROID_FEATURE_SUM;
        if (s == "feature_sum_pardim") return CLK_CENTROID_FEATURE_SUM_PARDIM;
        if (s == "cluster_merge") return CLK_CENTROID_CLUSTER_MERGE;
        break;
    default:
        set_error("clk_strategy_id: unknown stage");
        return CLK_ERR_INVALID_ARGUMENT;
    }
    set_error(s);  // the reference throws std::invalid_argument(strategy)
    return CLK_ERR_INVALID_ARGUMENT;
}

extern "C" int clk_default_config(clk_context *ctx, int stage, int strategy,
                                  clk_kernel_config *cfg)
{
    (void)ctx;
    CLK_REQUIRE(cfg != nullptr, CLK_ERR_INVALID_ARGUMENT, "clk_default_config: null cfg");
    std::memset(cfg, 0, sizeof(*cfg));
    cfg->stage = stage;
    cfg->strategy = strategy;
    cfg->local_size[0] = 256;
    cfg->local_size[1] = cfg->local_size[2] = 1;
    cfg->global_size[1] = cfg->global_size[2] = 1;
    cfg->global_size[0] = 0;  // persistent grid sized from occupancy
    cfg->vector_length = 4;
    cfg->local_features = 1;
    cfg->thread_features = 1;
    return CLK_OK;
}

extern "C" int clk_profiling_enable(clk_context *ctx, int enable)
{
    CLK_REQUIRE(ctx, CLK_ERR_INVALID_ARGUMENT, "null clk_context");
    ctx->profiling = enable != 0;
    return CLK_OK;
}

extern "C" int clk_profiling_set_iteration(clk_context *ctx, int iteration)
{
    CLK_REQUIRE(ctx, CLK_ERR_INVALID_ARGUMENT, "null clk_context");
    ctx->iteration = iteration;
    return CLK_OK;
}

extern "C" int clk_profiling_clear(clk_context *ctx)
{
    CLK_TRY(enter(ctx));
    for (auto &r : ctx->records) {
        (void)hipEventSynchronize(r.stop);
        ctx->event_pool.push_back(r.start);
        ctx->event_pool.push_back(r.stop);
    }
    ctx->records.clear();
    return CLK_OK;
}

extern "C" int64_t clk_profiling_count(clk_context *ctx)
{
    if (!ctx)
        return CLK_ERR_INVALID_ARGUMENT;
    return (int64_t)ctx->records.size();
}

extern "C" int clk_profiling_get(clk_context *ctx, int64_t i, char *name, size_t name_len,
                                 int32_t *iteration, float *ms)
{
    CLK_TRY(enter(ctx));
    CLK_REQUIRE(i >= 0 && (size_t)i < ctx->records.size(), CLK_ERR_INVALID_ARGUMENT,
                "clk_profiling_get: index out of range");
    TimingRecord &r = ctx->records[(size_t)i];
    if (name && name_len) {
        std::strncpy(name, r.name.c_str(), name_len - 1);
        name[name_len - 1] = '\0';
    }
    if (iteration)
        *iteration = r.iteration;
    if (ms) {
        CLK_HIP_CHECK(hipEventSynchronize(r.stop));
        CLK_HIP_CHECK(hipEventElapsedTime(ms, r.start, r.stop));
    }
    return CLK_OK;
}

extern "C" int clk_fill_zero(clk_context *ctx, void *ptr, uint64_t bytes, void *stream)
{
    CLK_TRY(enter(ctx));
    if (bytes == 0)
        return CLK_OK;
    CLK_REQUIRE(ptr != nullptr, CLK_ERR_INVALID_ARGUMENT, "clk_fill_zero: null pointer");
    hipStream_t s = as_stream(stream);
    uint8_t *p = static_cast<uint8_t *>(ptr);
    uint64_t head = 0;
    if (reinterpret_cast<uintptr_t>(p) % 16 != 0)
        head = bytes;  // unaligned: byte path for everything
    uint64_t n16 = head ? 0 : bytes / 16;
    uint8_t *tail = p + n16 * 16;
    uint64_t ntail = bytes - n16 * 16;
    uint64_t work = std::max(n16, ntail);
    unsigned grid = (unsigned)std::min<uint64_t>(div_up(work, 256), 4096);
    KernelTimer t(ctx, "Fill", s);
    hipLaunchKernelGGL(fill_zero_kernel, dim3(std::max(grid, 1u)), dim3(256), 0, s,
                       reinterpret_cast<uint4 *>(p), n16, tail, ntail);
    CLK_HIP_CHECK(hipGetLastError());
    return CLK_OK;
}

extern "C" int clk_init_first_x(clk_context *ctx, uint64_t d, uint64_t n, uint64_t k,
                                const float *points, float *centroids, void *stream)
{
    CLK_TRY(enter(ctx));
    CLK_REQUIRE(d >= 1 && n >= 1 && k >= 1, CLK_ERR_SIZE, "first_x: d, n, k must be >= 1");
    CLK_REQUIRE(points && centroids, CLK_ERR_INVALID_ARGUMENT, "first_x: null buffer");
    hipStream_t s = as_stream(stream);
    KernelTimer t(ctx, "FirstX", s);
    hipLaunchKernelGGL(first_x_kernel, dim3((unsigned)div_up(d * k, 256)), dim3(256), 0, s,
                       points, n, (uint32_t)d, (uint32_t)k, centroids);
    CLK_HIP_CHECK(hipGetLastError());
    return CLK_OK;
}

template <typename T>
static int matrix_add(clk_context *ctx, uint64_t count, T *fst, const T *snd, void *stream)
{
    CLK_TRY(enter(ctx));
    if (count == 0)
        return CLK_OK;
    CLK_REQUIRE(fst && snd, CLK_ERR_INVALID_ARGUMENT, "matrix_add: null buffer");
    hipStream_t s = as_stream(stream);
    unsigned grid = (unsigned)std::min<uint64_t>(div_up(count, 256), 8192);
    KernelTimer t(ctx, "MatrixBinaryOpMatrix", s);
    hipLaunchKernelGGL(matrix_add_kernel<T>, dim3(grid), dim3(256), 0, s, fst, snd, count);
    CLK_HIP_CHECK(hipGetLastError());
    return CLK_OK;
}

extern "C" int clk_matrix_add_u32(clk_context *ctx, uint64_t count, uint32_t *fst,
                                  const uint32_t *snd, void *stream)
{
    return matrix_add<uint32_t>(ctx, count, fst, snd, stream);
}

extern "C" int clk_matrix_add_f64(clk_context *ctx, uint64_t count, double *fst,
                                  const double *snd, void *stream)
{
    return matrix_add<double>(ctx, count, fst, snd, stream);
}

extern "C" int clk_reduce_vector_parcol_u32(clk_context *ctx, uint64_t num_cols,
                                            uint64_t result_rows, uint32_t *data,
                                            void *stream)
{
    CLK_TRY(enter(ctx));
    CLK_REQUIRE(num_cols >= 1, CLK_ERR_SIZE, "reduce_vector_parcol: num_cols must be >= 1");
    CLK_REQUIRE(data || result_rows == 0, CLK_ERR_INVALID_ARGUMENT, "reduce: null data");
    return launch_reduce_u32(ctx, data, num_cols, result_rows, data, as_stream(stream));
}

extern "C" int clk_reduce_vector_parcol_f64(clk_context *ctx, uint64_t num_cols,
                                            uint64_t result_rows, double *data,
                                            void *stream)
{
    CLK_TRY(enter(ctx));
    CLK_REQUIRE(num_cols >= 1, CLK_ERR_SIZE, "reduce_vector_parcol: num_cols must be >= 1");
    CLK_REQUIRE(data || result_rows == 0, CLK_ERR_INVALID_ARGUMENT, "reduce: null data");
    return launch_reduce_f64(ctx, data, num_cols, result_rows, data, as_stream(stream));
}

extern "C" int clk_matrix_divide_row(clk_context *ctx, uint64_t d, uint64_t k,
                                     const double *sums, const uint32_t *masses,
                                     float *centroids, const float *old_centroids,
                                     double *max_shift, void *stream)
{
    CLK_TRY(enter(ctx));
    CLK_REQUIRE(d >= 1 && k >= 1, CLK_ERR_SIZE, "divide: d and k must be >= 1");
    CLK_REQUIRE(d * k < (1ull << 32), CLK_ERR_SIZE, "divide: d*k too large");
    CLK_REQUIRE(sums && masses && centroids, CLK_ERR_INVALID_ARGUMENT, "divide: null buffer");
    CLK_REQUIRE(!old_centroids || old_centroids != centroids, CLK_ERR_INVALID_ARGUMENT,
                "divide: old_centroids must not alias centroids");
    hipStream_t s = as_stream(stream);
    KernelTimer t(ctx, "MatrixBinaryOpRow", s);
    if (!old_centroids || !max_shift) {
        hipLaunchKernelGGL(divide_values_kernel, dim3((unsigned)div_up(d * k, 256)), dim3(256), 0, s, sums, masses,
                           (uint32_t)(d * k), (uint32_t)k, centroids);
        CLK_HIP_CHECK(hipGetLastError());
        return CLK_OK;
    }
    unsigned block = 64;
    while (block < 1024 && block < k)
        block *= 2;  // power of two for the tree reduction
    hipLaunchKernelGGL(divide_kernel, dim3(1), dim3(block), 0, s, sums, masses, (uint32_t)d,
                       (uint32_t)k, centroids, old_centroids, max_shift);
    CLK_HIP_CHECK(hipGetLastError());
    return CLK_OK;
}
