// Labeling on the matrix cores with split operands: scores of about FP32
// accuracy from FP16 MFMA, so that few points need the exact scan.  One
// launch, no scratch memory: each work-group builds the operand table of the
// centroids in LDS.  The labels equal the sequential-fma scan's
// (lloyd_fused_feature_sum.cl:213-239, kmeans_naive.cpp:49-63) bit for bit.
//
// Scores.  Points and centroids are taken relative to a point m, the mean of
// eight centroids: below, x and c stand for x - m and c - m.  (Relative to the
// origin the scores of data far from it cancel, and nearly every point took
// the exact scan: 150k points d=11 k=300 around 300 labeling 703 -> 28 us, 3M
// d=8 k=64 126 -> 48; m costs about 1 us of every launch.)
// With a power of two s that puts max |c| into [2^12, 2^13), every coordinate
// is split into two FP16 parts: s x = xh + xl (toward zero), -2 s c = ch + cl
// (to nearest).  The MFMA accumulator starts at RN(||s c||^2), so S_c =
// ||s c||^2 - 2 s^2 x.c up to a bounded error.
// K = 32 of one 16x16x32 MFMA holds, for P padded features:
//   P = 4, 8 all four products xh ch, xh cl, xl ch, xl cl of the features;
//   P = 16   two MFMAs, (ch | cl) against (xh | xh) and (xl | xl);
//   P >= 32  three MFMAs per 32 features: xl ch, xh cl of all features from 0,
//            the norm added, then xh ch -- so that the small products are
//            summed while the sum is small, and round a third as much.
// Scores may be negative: they are ranked as floats.  A key is the score with
// its low bits replaced by an index.
//
// Error of one score (u = 2^-24, X >= ||s x|| over the padded features, C >= max ||s c||, N >= C^2):
//   split of x   Rx = 1.125 * 2^-20 X + 1.01 * 2^-24 sqrt(d)  (toward zero:
//                2^-10 relative per part, subnormal spacing 2^-24; and the
//                rounding of x - m, 2^-24 relative)
//   split of c   Rc = 1.3125 * 2^-22 2C + 1.01 * 2^-25 sqrt(d)  (with that of
//                c - m)
//   inputs       (X + Rx) Rc + Rx 2C; P >= 32 also the dropped xl cl:
//                (2^-10 X + 2^-24 sqrt(d)) (2^-11 2C + 2^-25 sqrt(d))
//   summation    g (N + 1.004 X 2C), g = 2(T+1)u / (1 - 2(T+1)u) for the T
//                products that are not padding (adding 0 is exact), each
//                addition rounding or truncating.  P >= 32: T = d (xh ch, on
//                top of the norm and the small products), the addition of the
//                norm 2u (N + their sum), and theirs, g' with T = 2d of
//                (2^-10 X + 2^-24 sqrt(d)) 2C (1 + 2^-11) + X (2^-11 2C + 2^-25 sqrt(d))
//   norm         4u N  (of coordinates rounded to FP32)
// E = 1.01 x the sum + a bound on flushed denormals.  An FP16 subnormal must
// reach the product: every launch checks that the matrix core keeps them, and
// without that every point takes the exact scan.
//
// Margin.  vb, vs: the two smallest keys; tr the relative key error 2^(bits -
// 23); e_c the reference's FP32 distance, within eps = (d+3)u relative (plus
// d 2^-125 absolute) of ||x-c||^2.  With D = vb + tr|vb| + E + X^2 >= the
// scaled ||x-c_b||^2,
//   vs - vb > 1.01 (2E + tr'(|vb| + |vs|) + 2.1 eps D + 2 s^2 d 2^-125),
// tr' = tr / (1 - tr),
// makes c_b the strict, unique minimum of e_c.  Every other point -- and every
// point with a coordinate that is not finite or too large for FP16 -- scans
// all centroids, or its candidates, with the reference's arithmetic: one by
// one (exact_scan, candidate_scan), or all points of the wave at once
// (scan_rows, block_scan), by what they cost.
//
// Double points (T = double): x - m and c - m are taken in FP64 and then
// rounded to FP32, one rounding as well; eps = (d+3) 2^-53 and the scans are
// FP64.
#pragma once

#include "clk_common.hpp"
#include "clk_mfma_device.hpp"

#include <type_traits>

namespace clk {
namespace split {

using mfma::f32v4;
using mfma::u16x8;

typedef __fp16 h16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

constexpr float kNever = 3.0e38f;  // norm of a padded or non-finite centroid

template <int P>
struct Shape {
    static constexpr int nkb = P < 32 ? 1 : P / 32;       // K-blocks of 32 features
    static constexpr int nops = P < 32 ? 1 : 2 * nkb;     // operand vectors per tile of 16 centroids
    static constexpr int terms = P < 32 ? 4 : 1;  // products per feature in the sum with the norm
    static constexpr int planes = P < 32 ? P / 4 : 0;  // LDS exchange, u16x8 [64] each
};

// LDS of one work-group of `waves` waves: table, norms, centroids as they are
// (P < 32: [k][P], 0 past d), m (past d that of feature d - 1), statistics,
// exchange.
template <int P>
__host__ __device__ constexpr size_t table_bytes(uint32_t ntiles)
{
    return (size_t)ntiles * Shape<P>::nops * 64 * sizeof(u16x8);
}
constexpr uint32_t kStatWords = 16;
template <int P, typename T>
__host__ __device__ constexpr size_t rows_bytes(uint32_t ntiles)
{
    return P < 32 ? (size_t)ntiles * 16 * P * sizeof(T) : 0;
}
template <int P, typename T>
__host__ __device__ constexpr size_t lds_bytes(uint32_t ntiles, uint32_t waves)
{
    return table_bytes<P>(ntiles) + rows_bytes<P, T>(ntiles) + (size_t)ntiles * 16 * sizeof(float) + P * sizeof(T) +
           kStatWords * sizeof(float) +
           (size_t)waves * Shape<P>::planes * 64 * sizeof(u16x8);
}

__device__ __forceinline__ float min_f(float a, float b)
{
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float max_f(float a, float b)
{
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float min3_f(float a, float b, float c)
{
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float med3_f(float a, float b, float c)
{
    float r;
    asm("v_med3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Two keys into (best, second): the two smallest of the four.
__device__ __forceinline__ void push2(float &best, float &second, float a, float b)
{
    const float m = med3_f(best, a, b);
    best = min3_f(best, a, b);
    second = min_f(second, m);
}

__device__ __forceinline__ void merge_pair(float &b, float &s, float b2, float s2)
{
    s = min3_f(max_f(b, b2), s, s2);
    b = min_f(b, b2);
}

// Swap the upper half-wave of a with the lower half-wave of b / the odd rows
// of 16 lanes of a with the even rows of b.
__device__ __forceinline__ void swap32(float &a, float &b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap16(float &a, float &b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}

// What the work-group's table says, wave-uniform.
template <typename T>
struct Table {
    const u16x8 *ops;
    const float *norm;
    const T *rows;
    const T *mean;  // m
    uint32_t ntiles, kmask;
    float scale;    // s
    // the margin: t0 + tX ||s x|| + tx2 ||s x||^2 + tk (|vb| + |vs|)
    float t0, tX, tx2, tk;
    bool ok;
};

// The margin's coefficients (see the header; each is rounded up by far more
// than the rounding of its evaluation and of the margin's).
template <int P, typename T>
__device__ __forceinline__ void set_margin(Table<T> &t, float N, uint32_t d, uint32_t bits)
{
    constexpr bool f64 = sizeof(T) == 8;
    constexpr float up = 1.0f + 1e-4f;
    const float C2 = 2.0f * sqrtf(N) * up, sd = sqrtf((float)d) * up;
    const float terms = (float)(Shape<P>::terms * d);
    const float g0 = 2.0f * (terms + 1.0f) * mfma::kU;
    const float gamma = g0 / (1.0f - g0) * up;
    constexpr float alpha = 0x1.2p-20f;
    const float beta = 1.01f * 0x1p-24f * sd;
    const float Rc = 0x1.5p-22f * C2 + 1.01f * 0x1p-25f * sd;
    float e1 = (1.0f + alpha) * Rc + alpha * C2 + gamma * 1.004f * C2;
    float e0 = beta * (Rc + C2) + (gamma + 4.0f * mfma::kU) * N;
    if constexpr (P >= 32) {
        const float m = 0x1p-11f * C2 + 0x1p-25f * sd;
        e1 += 0x1p-10f * m;
        e0 += 0x1p-24f * sd * m;
        // the small products' sum is at most s1 X + s0; g2 their summation,
        // the norm's addition to it and its part in the last one
        const float s1 = 1.01f * (0x1p-10f * C2 + m), s0 = 1.01f * 0x1p-24f * sd * C2;
        const float g2 = 4.0f * ((float)d + 1.0f) * mfma::kU / (1.0f - 4.0f * ((float)d + 1.0f) * mfma::kU) * up +
                         2.0f * mfma::kU + gamma;
        e1 += g2 * s1;
        e0 += g2 * s0 + 2.0f * mfma::kU * N;
    }
    e1 *= 1.01f;
    e0 = 1.01f * e0 + (4.0f * (float)d + 2.0f) * 0x1p-125f;
    const float eps = (float)(d + 3) * (f64 ? 0x1p-53f : mfma::kU) * up;
    const float tr0 = __uint_as_float((bits - 23 + 127) << 23), tr = tr0 / (1.0f - tr0) * up;
    const float under = f64 ? 0.0f : t.scale * t.scale * (float)d * 0x1p-125f;
    t.t0 = up * (1.01f * ((2.0f + 2.1f * eps) * e0 + 2.0f * under) + 1e-30f);
    t.tX = up * 1.01f * (2.0f + 2.1f * eps) * e1;
    t.tx2 = up * 1.01f * 2.1f * eps;
    t.tk = up * 1.01f * (tr + 2.1f * eps * (1.0f + tr));
}

// Build the table of cen [d][k] (whole work-group; ends with a barrier).
template <int P, typename T>
__device__ __forceinline__ Table<T> stage(const T *__restrict__ cen, uint32_t d, uint32_t k, uint32_t ntiles,
                                          char *lds)
{
    using Sh = Shape<P>;
    constexpr bool f64 = sizeof(T) == 8;
    constexpr T kMax = f64 ? (T)DBL_MAX : (T)FLT_MAX;
    Table<T> t;
    u16x8 *ops = reinterpret_cast<u16x8 *>(lds);
    float *norm = reinterpret_cast<float *>(lds + table_bytes<P>(ntiles));
    T *rows = reinterpret_cast<T *>(norm + ntiles * 16);
    T *mean = reinterpret_cast<T *>(reinterpret_cast<char *>(rows) + rows_bytes<P, T>(ntiles));
    uint32_t *stat = reinterpret_cast<uint32_t *>(mean + P);
    const uint32_t tid = threadIdx.x, B = blockDim.x, dk = d * k;
    if (tid < kStatWords)
        stat[tid] = 0;
    // m: the mean of 8 centroids (an eighth of each: no sum overflows)
    constexpr uint32_t kSample = 8, kFirst = 4;
    T first[kFirst];  // of the next pass, loaded with them
#pragma unroll
    for (uint32_t j = 0; j < kFirst; ++j)
        first[j] = cen[min(tid + j * B, dk - 1)];
    if (tid < P) {
        T sum = 0;
#pragma unroll
        for (uint32_t j = 0; j < kSample; ++j) {
            const T v = cen[min(tid, d - 1) * k + j * k / kSample];
            sum += __builtin_fabs(v) <= kMax ? v * (T)(1.0 / kSample) : (T)0;
        }
        mean[tid] = sum;
    }
    __syncthreads();
    // stat[0]: max |c - m| over the finite coordinates; beyond FP32 its largest
    // value, which no scale takes
    uint32_t m = 0;
    const float per_row = 1.0f / (float)k;
    // i / k: i < 2^18, so the product is off by less than the half added
    auto row_of = [&](uint32_t i) { return (uint32_t)(((float)i + 0.5f) * per_row); };
    auto take = [&](T v, uint32_t i) {
        const T a = v - mean[row_of(i)];
        const uint32_t u = min(__float_as_uint(__builtin_fabsf((float)a)), 0x7F7FFFFFu);
        m = (__builtin_fabs(v) <= kMax && u > m) ? u : m;
    };
#pragma unroll
    for (uint32_t j = 0; j < kFirst; ++j)
        if (tid + j * B < dk)
            take(first[j], tid + j * B);
#pragma unroll 2
    for (uint32_t i = tid + kFirst * B; i < dk; i += B)
        take(cen[i], i);
    for (int o = 32; o >= 1; o /= 2)
        m = max(m, (uint32_t)__shfl_xor((int)m, o));
    if (tid % 64 == 0 && m)
        atomicMax(&stat[0], m);
    __syncthreads();
    const int ex = max((int)(stat[0] >> 23) - 127, -88);  // max |c| < 2^(ex + 1)
    t.ok = ex <= 56;  // distances of points that FP16 holds stay far below FLT_MAX
    const float s = __uint_as_float((uint32_t)(12 - (t.ok ? ex : 0) + 127) << 23);
    t.scale = s;
    for (uint32_t e = tid; e < ntiles * Sh::nops * 64; e += B) {
        const uint32_t lane = e % 64, op = (e / 64) % Sh::nops, tile = e / (64 * Sh::nops);
        const uint32_t c = tile * 16 + lane % 16, h = lane / 16;
        const bool low = P == 8 ? (h & 1) != 0 : P == 16 ? h >= 2 : (op & 1) != 0;
        const uint32_t f0 = P <= 8 ? 0 : P == 16 ? 8 * (h & 1) : (op / 2) * 32 + 8 * h;
        u16x8 v;
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
            // P = 4: (ch | cl) in the first two quarters, zeros in the others
            const uint32_t f = P == 4 ? j % 4 : f0 + j;
            const bool lo = P == 4 ? j >= 4 : low;
            const T raw = cen[min(f * k + c, dk - 1)];
            const bool in = c < k && f < d && (P != 4 || h < 2) && __builtin_fabs(raw) <= kMax;
            float x = in ? -2.0f * s * (float)(T)(raw - mean[f]) : 0.0f;
            // both parts come from the FP32 value: the compiler would round a
            // double to FP16 at once for the high part, and not to the same
            // neighbour when the FP32 value lies between two
            asm("" : "+v"(x));
            _Float16 p = (_Float16)x;
            if (lo)
                p = (_Float16)(x - (float)p);
            v[j] = __builtin_bit_cast(uint16_t, p);
        }
        ops[e] = v;
    }
    if constexpr (P < 32)
        for (uint32_t i = tid; i < k * P; i += B) {
            const uint32_t f = row_of(i), c = i - f * k;
            rows[c * P + f] = f < d ? cen[min(i, dk - 1)] : (T)0;
        }
    uint32_t nmax = 0;
    for (uint32_t c = tid; c < ntiles * 16; c += B) {
        double q = 0.0;
        bool fin = c < k;
#pragma unroll 8
        for (uint32_t f = 0; f < d; ++f) {
            const T v = cen[min(f * k + c, dk - 1)];
            fin = fin && __builtin_fabs(v) <= kMax;
            const double w = f64 ? (double)(v - mean[f]) * (double)s : (double)((float)(v - mean[f]) * s);
            q = __builtin_fma(w, w, q);
        }
        norm[c] = fin ? (float)q : kNever;
        const uint32_t u = __float_as_uint((float)(q * (1.0 + 1e-6)));
        nmax = fin && u > nmax ? u : nmax;
    }
    for (int o = 32; o >= 1; o /= 2)
        nmax = max(nmax, (uint32_t)__shfl_xor((int)nmax, o));
    if (tid % 64 == 0 && nmax)
        atomicMax(&stat[1], nmax);
    {  // does the matrix core keep FP16 subnormals?  32 x 2^-20 x 1
        u16x8 a, b;
        for (int j = 0; j < 8; ++j) {
            a[j] = mfma::to16<true>(0x1p-20f);
            b[j] = mfma::to16<true>(1.0f);
        }
        const f32v4 r = mfma::mma16<true>(a, b, f32v4{0.0f, 0.0f, 0.0f, 0.0f});
        t.ok = t.ok && r[0] == 0x1p-15f;
    }
    __syncthreads();
    t.ops = ops;
    t.norm = norm;
    t.rows = rows;
    t.mean = mean;
    t.ntiles = ntiles;
    uint32_t bits = 4;
    while ((1u << bits) < ntiles * 16)
        ++bits;
    t.kmask = (1u << bits) - 1u;
    set_margin<P, T>(t, __uint_as_float(stat[1]), d, bits);
    return t;
}

// Two scaled coordinates -> their high and low FP16 parts, packed.
__device__ __forceinline__ void split2(float a, float b, uint32_t &hi, uint32_t &lo)
{
    const h16x2 h = __builtin_amdgcn_cvt_pkrtz(a, b);
    const h16x2 l = __builtin_amdgcn_cvt_pkrtz(a - (float)h[0], b - (float)h[1]);
    hi = __builtin_bit_cast(uint32_t, h);
    lo = __builtin_bit_cast(uint32_t, l);
}

// The wave's 64 points as B operands, four groups of 16.
template <int P>
struct PointOps {
    u16x8 hi[4][Shape<P>::nkb];
    u16x8 lo[P <= 8 ? 1 : 4][Shape<P>::nkb];  // P <= 8: hi holds both parts
};

// P <= 16: lane = point, coordinates x (past d any of
// the point's coordinates again: the centroids are 0 there).  buf: this wave's
// exchange planes.  Returns a bound >= ||s x||^2.
template <int P, typename T>
__device__ __forceinline__ float build_points(const Table<T> &t, const T (&x)[P], u16x8 *buf, uint32_t lane,
                                              PointOps<P> &o)
{
    static_assert(P < 32, "lane = point form");
    float x2 = 0.0f;
    uint32_t hi[P / 2], lo[P / 2];
#pragma unroll
    for (int f = 0; f < P; f += 2) {
        const float a = (float)(x[f] - t.mean[f]) * t.scale, b = (float)(x[f + 1] - t.mean[f + 1]) * t.scale;
        x2 = __builtin_fmaf(a, a, x2);
        x2 = __builtin_fmaf(b, b, x2);
        split2(a, b, hi[f / 2], lo[f / 2]);
    }
    const uint32_t q = lane % 16, h = lane / 16;
    mfma::wave_lds_order();  // the previous step's reads are done
    if constexpr (P == 4) {
        buf[lane] = __builtin_bit_cast(u16x8, v4u{hi[0], hi[1], lo[0], lo[1]});
        mfma::wave_lds_order();
        typedef uint32_t v2u __attribute__((ext_vector_type(2)));
        const v2u *half = reinterpret_cast<const v2u *>(buf);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const v2u w = half[(g * 16 + q) * 2 + (h & 1)];
            o.hi[g][0] = __builtin_bit_cast(u16x8, v4u{w.x, w.y, w.x, w.y});
        }
    } else {
#pragma unroll
        for (int i = 0; i < P / 8; ++i) {
            buf[i * 64 + lane] = __builtin_bit_cast(u16x8, v4u{hi[4 * i], hi[4 * i + 1], hi[4 * i + 2], hi[4 * i + 3]});
            buf[(P / 8 + i) * 64 + lane] =
                __builtin_bit_cast(u16x8, v4u{lo[4 * i], lo[4 * i + 1], lo[4 * i + 2], lo[4 * i + 3]});
        }
        mfma::wave_lds_order();
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if constexpr (P == 8) {
                o.hi[g][0] = buf[(h / 2) * 64 + g * 16 + q];
            } else {
                o.hi[g][0] = buf[(h & 1) * 64 + g * 16 + q];
                o.lo[g][0] = buf[(2 + (h & 1)) * 64 + g * 16 + q];
            }
        }
    }
    return x2 * (1.0f + (float)(2 * P + 12) * mfma::kU);
}

// P >= 32: lane (q, h) holds raw[g][kb*8 + j] = feature kb*32 + 8h + j of
// point g*16 + q (past d as above).  Returns a bound >= ||s x||^2 of this
// lane's own point (lane 16h + q).
template <int P, typename T>
__device__ __forceinline__ float build_points(const Table<T> &t, const T (&raw)[4][Shape<P>::nkb * 8], uint32_t lane,
                                              PointOps<P> &o)
{
    static_assert(P >= 32, "matrix layout");
    float mine = 0.0f;
    const T *const mean = t.mean + 8 * (lane / 16);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        float x2 = 0.0f;
#pragma unroll
        for (int kb = 0; kb < Shape<P>::nkb; ++kb) {
            v4u hi, lo;
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                const float a = (float)(raw[g][kb * 8 + j] - mean[kb * 32 + j]) * t.scale;
                const float b = (float)(raw[g][kb * 8 + j + 1] - mean[kb * 32 + j + 1]) * t.scale;
                x2 = __builtin_fmaf(a, a, x2);
                x2 = __builtin_fmaf(b, b, x2);
                uint32_t h, l;
                split2(a, b, h, l);
                hi[j / 2] = h;
                lo[j / 2] = l;
            }
            o.hi[g][kb] = __builtin_bit_cast(u16x8, hi);
            o.lo[g][kb] = __builtin_bit_cast(u16x8, lo);
        }
        x2 += mfma::xor_swizzle<16>(x2);
        x2 += __shfl_xor(x2, 32);
        mine = (uint32_t)g == lane / 16 ? x2 : mine;
    }
    return mine * (1.0f + (float)(2 * P + 12) * mfma::kU);
}

// The scores of a tile: acc[g][i] of point 16g + q and centroid 16 tile + 4h + i.
template <int P, typename T>
__device__ __forceinline__ void score_tile(const Table<T> &t, const PointOps<P> &x, uint32_t tile, uint32_t lane,
                                           f32v4 (&acc)[4])
{
    using Sh = Shape<P>;
    const f32v4 nrm = *reinterpret_cast<const f32v4 *>(t.norm + tile * 16 + 4 * (lane / 16));
    if constexpr (P < 32) {
        const u16x8 a = t.ops[tile * 64 + lane];
#pragma unroll
        for (int g = 0; g < 4; ++g)
            acc[g] = mfma::mma16<true>(a, x.hi[g][0], nrm);
        if constexpr (P == 16)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                acc[g] = mfma::mma16<true>(a, x.lo[g][0], acc[g]);
    } else {
        u16x8 ah[Sh::nkb];
#pragma unroll
        for (int kb = 0; kb < Sh::nkb; ++kb) {
            ah[kb] = t.ops[(tile * Sh::nops + 2 * kb) * 64 + lane];
            const u16x8 al = t.ops[(tile * Sh::nops + 2 * kb + 1) * 64 + lane];
#pragma unroll
            for (int g = 0; g < 4; ++g)
                acc[g] = mfma::mma16<true>(ah[kb], x.lo[g][kb], kb == 0 ? f32v4{0.0f, 0.0f, 0.0f, 0.0f} : acc[g]);
#pragma unroll
            for (int g = 0; g < 4; ++g)
                acc[g] = mfma::mma16<true>(al, x.hi[g][kb], acc[g]);
        }
#pragma unroll
        for (int g = 0; g < 4; ++g)
            acc[g] += nrm;
#pragma unroll
        for (int kb = 0; kb < Sh::nkb; ++kb)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                acc[g] = mfma::mma16<true>(ah[kb], x.hi[g][kb], acc[g]);
    }
}

// The two smallest keys of this lane's own point over all centroids.  A key's
// low bits hold (4 tile + i) * 4 + h for row 4h + i of a tile: the tile and
// row parts are the same for all lanes (scalar operands), h is put in once
// after the last tile; centroid_of undoes it.
__device__ __forceinline__ uint32_t centroid_of(float key, uint32_t kmask)
{
    const uint32_t l = __float_as_uint(key) & kmask;
    return (l & ~15u) | ((l & 3u) << 2) | ((l >> 2) & 3u);
}

template <int P, typename T>
__device__ __forceinline__ void rank_points(const Table<T> &t, const PointOps<P> &x, uint32_t lane, float &best,
                                            float &second)
{
    const uint32_t h = lane / 16;
    float b[4], s[4];
#pragma unroll
    for (int g = 0; g < 4; ++g)
        b[g] = s[g] = FLT_MAX;
    const uint32_t vkeep = mfma::opaque_v(~t.kmask);
    for (uint32_t tile = 0; tile < t.ntiles; ++tile) {
        f32v4 acc[4];
        score_tile<P>(t, x, tile, lane, acc);
        uint32_t idx[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            idx[i] = mfma::opaque_s((4 * tile + i) * 4);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            float key[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                key[i] = __uint_as_float((__float_as_uint(acc[g][i]) & vkeep) | idx[i]);
            push2(b[g], s[g], key[0], key[1]);
            push2(b[g], s[g], key[2], key[3]);
        }
    }
#pragma unroll
    for (int g = 0; g < 4; ++g)
        b[g] = __uint_as_float(__float_as_uint(b[g]) | h);
    // The four lanes of a column hold the four row quarters of every group:
    // after two exchanges lane row h holds group h, merged.
    swap32(b[0], b[2]);
    swap32(s[0], s[2]);
    merge_pair(b[0], s[0], b[2], s[2]);
    swap32(b[1], b[3]);
    swap32(s[1], s[3]);
    merge_pair(b[1], s[1], b[3], s[3]);
    swap16(b[0], b[1]);
    swap16(s[0], s[1]);
    merge_pair(b[0], s[0], b[1], s[1]);
    best = b[0];
    second = s[0];
}

// Margin test of this lane's own point; lab = the best key's centroid.  limit:
// a centroid whose key v has v - t.tk |v| > limit is farther than the best
// key's by the reference's arithmetic (NaN, which nothing exceeds, where the
// bounds do not hold).
template <typename T>
__device__ __forceinline__ bool decide(const Table<T> &t, float x2, float best, float second, uint32_t k, uint32_t &lab,
                                       float &limit)
{
    const float X = __builtin_amdgcn_sqrtf(x2);  // within one ulp
    const float ab = __builtin_fabsf(best);
    float base = __builtin_fmaf(t.tX, X, t.t0);
    base = __builtin_fmaf(t.tx2, x2, base);
    const float tau = __builtin_fmaf(t.tk, ab + __builtin_fabsf(second), base);
    lab = centroid_of(best, t.kmask);
    // NaN fails every test; 4.2e9 < 65504^2; a key of denormal size is not
    // trusted to keep its index
    const bool holds = t.ok && x2 < 4.2e9f && best < 1e37f && ab > 1e-30f && lab < k;
    base = __builtin_fmaf(t.tk, ab, base);
    // rounded up: by more than this sum's and the test's own roundings
    limit = holds ? best + base + 8.0f * mfma::kU * (ab + base) : __builtin_nanf("");
    return holds && second - best > tau;
}

// The reference's scan, over all centroids, of the wave's points whose bit is
// set in open: 64 / G points at a time, G lanes each (8 <= G <= 64, a lane per
// centroid while k <= G), up to sixteen features' loads in flight.  base: the
// coordinate of feature 0 of the wave's point 0, the rows n apart.  lab of
// lane i becomes the label of point i.
template <int P, typename T>
__device__ __forceinline__ void exact_scan(uint64_t open, const T *__restrict__ base, uint64_t n,
                                           const T *__restrict__ cen, uint32_t d, uint32_t k, uint32_t lane,
                                           uint32_t &lab)
{
    constexpr bool f64 = sizeof(T) == 8;
    constexpr T kMax = f64 ? (T)DBL_MAX : (T)FLT_MAX;
    constexpr uint32_t kAhead = P == 4 ? 4 : f64 ? 8 : 16;
    uint32_t G = 8;
    while (G < k && G < 64)
        G *= 2;
    while (open) {
        uint64_t rest = open;
        uint32_t src = 0;  // this lane's point
        for (uint32_t i = 0; i < 64 / G && rest; ++i) {
            const uint32_t bit = (uint32_t)__builtin_ctzll(rest);
            rest &= rest - 1;
            src = lane / G >= i ? bit : src;  // groups past the last point repeat it
        }
        const T *x = base + src;
        T best = kMax;
        uint32_t bi = 0;
        for (uint32_t c0 = 0; c0 < k; c0 += G) {
            const uint32_t c = c0 + lane % G;
            const T *col = cen + min(c, k - 1);
            T dist = 0;
            for (uint32_t f0 = 0; f0 < d; f0 += kAhead) {
                T xv[kAhead], cv[kAhead];
#pragma unroll
                for (uint32_t j = 0; j < kAhead; ++j) {
                    const uint32_t f = min(f0 + j, d - 1);
                    xv[j] = x[(uint64_t)f * n];
                    cv[j] = col[(size_t)f * k];
                }
#pragma unroll
                for (uint32_t j = 0; j < kAhead; ++j)
                    if (f0 + j < d) {
                        const T u = xv[j] - cv[j];
                        if constexpr (f64)
                            dist = __builtin_fma(u, u, dist);
                        else
                            dist = __builtin_fmaf(u, u, dist);
                    }
            }
            if (c < k && dist < best) {
                best = dist;
                bi = c;
            }
        }
        // smallest distance, lowest index on equal distances; none below the
        // largest value gives label 0
        for (uint32_t o = G / 2; o >= 1; o /= 2) {
            const T b2 = __shfl_xor(best, (int)o);
            const uint32_t i2 = (uint32_t)__shfl_xor((int)bi, (int)o);
            const bool take = b2 < best || (b2 == best && i2 < bi);
            best = take ? b2 : best;
            bi = take ? i2 : bi;
        }
        const uint32_t found = best < kMax ? bi : 0u;
        for (uint32_t i = 0; i < 64 / G && open; ++i) {
            const uint32_t bit = (uint32_t)__builtin_ctzll(open);
            open &= open - 1;
            const uint32_t r = (uint32_t)__builtin_amdgcn_readlane((int)found, (int)(i * G));
            lab = lane == bit ? r : lab;
        }
    }
}

// Lane I of this lane's row of 16.
template <int I, typename T>
__device__ __forceinline__ T row_lane(T v)
{
    constexpr int kRowNewBcast = 0x150;
    if constexpr (sizeof(T) == 8)
        return __builtin_amdgcn_update_dpp(v, v, kRowNewBcast + I, 0xf, 0xf, true);
    else
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), kRowNewBcast + I, 0xf, 0xf, true));
}

template <int I, int CB, typename T>
__device__ __forceinline__ void add_squares(T xv, T cv, T (&dist)[CB])
{
    const T u = row_lane<I>(cv) - xv;  // the square of x - c, whichever its sign
    if constexpr (sizeof(T) == 8)
        dist[I] = __builtin_fma(u, u, dist[I]);
    else
        dist[I] = __builtin_fmaf(u, u, dist[I]);
    if constexpr (I + 1 < CB)
        add_squares<I + 1, CB>(xv, cv, dist);
}

// The reference's scan, over all centroids, of all the wave's points: lane =
// point (x: its feature 0, the rows n apart), 16 centroids at a time, one in
// every lane of each row of 16 lanes, from where the subtraction broadcasts
// it; the loads four features ahead.  Vector operations bound it, 2 k d for
// the 64 points, where exact_scan takes 2 d loads for each point and 64
// centroids: it is the faster one from about six points on (1M equal points
// d=20 k=130, double, labeling 4185 -> 409 us; 1M d=32 k=64 out of the scores'
// range 1351 -> 191, the plain kernel 113).
template <typename T>
__device__ __forceinline__ uint32_t block_scan(const T *__restrict__ x, uint64_t n, const T *__restrict__ cen,
                                               uint32_t d, uint32_t k, uint32_t lane)
{
    constexpr int kBlock = 16;
    constexpr uint32_t kAhead = 4;
    T best = sizeof(T) == 8 ? (T)DBL_MAX : (T)FLT_MAX;
    uint32_t lab = 0;
    for (uint32_t c0 = 0; c0 < k; c0 += kBlock) {
        const T *const col = cen + min(c0 + lane % kBlock, k - 1);  // the last centroid again: never less than itself
        T dist[kBlock], xv[kAhead], cv[kAhead];
#pragma unroll
        for (int i = 0; i < kBlock; ++i)
            dist[i] = 0;
        auto load = [&](uint32_t j, uint32_t f) {
            xv[j] = x[(uint64_t)min(f, d - 1) * n];
            cv[j] = col[(size_t)min(f, d - 1) * k];
        };
#pragma unroll
        for (uint32_t j = 0; j < kAhead; ++j)
            load(j, j);
        uint32_t f = 0;
        for (; f + kAhead <= d; f += kAhead)
#pragma unroll
            for (uint32_t j = 0; j < kAhead; ++j) {
                add_squares<0, kBlock>(xv[j], cv[j], dist);
                load(j, f + kAhead + j);
            }
#pragma unroll
        for (uint32_t j = 0; j < kAhead - 1; ++j)
            if (f + j < d)
                add_squares<0, kBlock>(xv[j], cv[j], dist);
#pragma unroll
        for (int i = 0; i < kBlock; ++i)
            if (dist[i] < best) {
                best = dist[i];
                lab = c0 + i;
            }
    }
    return lab;
}

// The points of open settled among the centroids that their limits leave
// (usually two or three): the tiles are scored again, and every lane takes the
// exact distances of its rows' candidates, its own point and centroid each.
// base as in exact_scan.  false, with lab as it was: a lane has more than six
// candidates in a tile, the scan of all centroids is the cheaper one.
template <int P, typename T>
__device__ __forceinline__ bool candidate_scan(const Table<T> &t, const PointOps<P> &ops, uint64_t open, float limit,
                                               const T *__restrict__ base, uint64_t n, const T *__restrict__ cen,
                                               uint32_t d, uint32_t k, uint32_t lane, uint32_t &lab)
{
    constexpr bool f64 = sizeof(T) == 8;
    constexpr T kMax = f64 ? (T)DBL_MAX : (T)FLT_MAX;
    constexpr uint32_t kAhead = f64 || P > 64 ? 8 : 16;
    const uint32_t q = lane % 16, h = lane / 16;
    float lim[4];
    T best[4];
    uint32_t at[4];
    uint32_t live = 0;  // bits 4g .. 4g+3: this lane's point of group g is open
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        lim[g] = __shfl(limit, g * 16 + (int)q);
        live |= (open >> (g * 16 + q)) & 1 ? 15u << (4 * g) : 0u;
        best[g] = kMax;
        at[g] = 0;
    }
    for (uint32_t tile = 0; tile < t.ntiles; ++tile) {
        f32v4 acc[4];
        score_tile<P>(t, ops, tile, lane, acc);
        uint32_t cand = 0;
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // the score itself: its key is within t.tk of it
                const float v = acc[g][i];
                const bool in = v - 2.0f * t.tk * __builtin_fabsf(v) <= lim[g] && tile * 16 + 4 * h + i < k;
                cand |= (in ? 1u : 0u) << (4 * g + i);
            }
        cand &= live;
        if (__ballot(__builtin_popcount(cand) > 6))
            return false;
        while (cand) {
            const uint32_t bit = (uint32_t)__builtin_ctz(cand), g = bit / 4;
            cand &= cand - 1;
            const uint32_t c = tile * 16 + 4 * h + bit % 4;
            const T *x = base + g * 16 + q, *col = cen + c;
            T dist = 0;
            for (uint32_t f0 = 0; f0 < d; f0 += kAhead) {
                T xv[kAhead], cv[kAhead];
#pragma unroll
                for (uint32_t j = 0; j < kAhead; ++j) {
                    const uint32_t f = min(f0 + j, d - 1);
                    xv[j] = x[(uint64_t)f * n];
                    cv[j] = col[(size_t)f * k];
                }
#pragma unroll
                for (uint32_t j = 0; j < kAhead; ++j)
                    if (f0 + j < d) {
                        const T u = xv[j] - cv[j];
                        if constexpr (f64)
                            dist = __builtin_fma(u, u, dist);
                        else
                            dist = __builtin_fmaf(u, u, dist);
                    }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)  // ascending centroids: strict
                if ((uint32_t)i == g && dist < best[i]) {
                    best[i] = dist;
                    at[i] = c;
                }
        }
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        T b = best[g];
        uint32_t c = at[g];
        for (int o = 16; o <= 32; o *= 2) {
            const T b2 = __shfl_xor(b, o);
            const uint32_t c2 = (uint32_t)__shfl_xor((int)c, o);
            const bool take = b2 < b || (b2 == b && c2 < c);
            b = take ? b2 : b;
            c = take ? c2 : c;
        }
        if ((uint32_t)g == h && ((open >> lane) & 1))
            lab = c;
    }
    return true;
}

// The reference's scan of this lane's own point x over the staged rows.
template <int P, typename T>
__device__ __forceinline__ uint32_t scan_rows(const Table<T> &t, const T (&x)[P], uint32_t d, uint32_t k)
{
    T best = sizeof(T) == 8 ? (T)DBL_MAX : (T)FLT_MAX;
    uint32_t lab = 0;
    T own[P];
    const uint32_t dd = mfma::opaque_s(d);  // no tests kept in scalar registers
#pragma unroll
    for (int f = 0; f < P; ++f)
        own[f] = f < (int)dd ? x[f] : (T)0;
    for (uint32_t c = 0; c < k; ++c) {
        const T *row = t.rows + c * P;
        T dist = 0;
#pragma unroll
        for (int f = 0; f < P; ++f) {  // 0 past d: adds fma(0, 0, dist) == dist
            const T u = own[f] - row[f];
            if constexpr (sizeof(T) == 8)
                dist = __builtin_fma(u, u, dist);
            else
                dist = __builtin_fmaf(u, u, dist);
        }
        const bool lt = dist < best;
        best = lt ? dist : best;
        lab = lt ? c : lab;
    }
    return lab;
}

}  // namespace split
}  // namespace clk
