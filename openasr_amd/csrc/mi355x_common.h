// mi355x_common.h -- shared definitions for the gfx950 backend: error
// handling, tensor views passed to kernels, block formats and device helpers.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>

#include "ggml_abi.h"

#define MI_CHECK(expr)                                                                                   \
    do {                                                                                                 \
        hipError_t err__ = (expr);                                                                       \
        if (err__ != hipSuccess) {                                                                       \
            std::fprintf(stderr, "mi355x: %s failed at %s:%d: %s\n", #expr, __FILE__, __LINE__,         \
                         hipGetErrorString(err__));                                                      \
            mi355x::note_hip_error(err__);                                                               \
        }                                                                                                \
    } while (0)

namespace mi355x {

void note_hip_error(hipError_t err);

constexpr int kWave = 64;

// A tensor as a kernel sees it: base pointer plus element counts and byte
// strides in ggml order (dim 0 innermost).
struct tview {
    char * data;
    int64_t ne[4];
    int64_t nb[4];
};

inline tview make_view(const ggml_tensor * t) {
    tview v;
    v.data = (char *) t->data;
    for (int i = 0; i < 4; i++) {
        v.ne[i] = t->ne[i];
        v.nb[i] = (int64_t) t->nb[i];
    }
    return v;
}

// Q8_0 weights are stored per row as [K int8 quants][K/32 f16 scales]
// (same byte count as ggml's interleaved 34-byte blocks) so a lane can issue
// aligned 16-byte loads of quants. Conversion happens in set/get_tensor.
inline size_t q8_0_row_bytes(int64_t k) { return (size_t) (k / 32) * 34; }

// Activations quantized for a Q8_0 weight: per column K int8 + K/32 f32
// scales (the f32 value of the f16-rounded scale ggml stores).
// Activations quantized for a Q4_K weight (ggml's Q8_K): per column K int8,
// K/256 f32 scales and K/16 int16 partial sums.
struct act_layout {
    int64_t q_stride;   // bytes between columns of quants
    int64_t d_stride;   // floats between columns of scales
    int64_t ss_stride;  // int16 between columns of 32-element sums (Q8_K only)
};

__device__ __forceinline__ float half_bits_to_float(uint16_t h) {
    return __half2float(__ushort_as_half(h));
}

__device__ __forceinline__ uint16_t float_to_half_bits(float f) {
    return __half_as_ushort(__float2half_rn(f));
}

__device__ __forceinline__ float round_to_half(float f) { return __half2float(__float2half_rn(f)); }

__device__ __forceinline__ int dot4_i8(int a, int b, int c) { return __builtin_amdgcn_sdot4(a, b, c, false); }

template <int W>
__device__ __forceinline__ float group_sum(float v) {
#pragma unroll
    for (int off = W / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, W);
    return v;
}

template <int W>
__device__ __forceinline__ float group_max(float v) {
#pragma unroll
    for (int off = W / 2; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, W));
    return v;
}

__device__ __forceinline__ float wave_sum(float v) { return group_sum<kWave>(v); }
__device__ __forceinline__ float wave_max(float v) { return group_max<kWave>(v); }

__device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// exp and sin/cos as a fixed sequence of IEEE double operations rounded once
// to f32 (the library is built without FMA contraction). The CPU reference
// evaluates the identical sequence, so host and device agree bit for bit and
// both are within one rounding of the exact value.
__device__ __forceinline__ float expf_det(float x) {
    if (x != x) return x;
    if (x > 88.72284f) return INFINITY;
    if (x < -103.97208f) return 0.0f;
    const double xd = (double) x;
    const double k = rint(xd * 1.4426950408889634074);
    const double r = (xd - k * 0.69314718055994528623) - k * 2.3190468138462996154e-17;
    double p = 1.0 / 479001600.0;
    p = p * r + 1.0 / 39916800.0;
    p = p * r + 1.0 / 3628800.0;
    p = p * r + 1.0 / 362880.0;
    p = p * r + 1.0 / 40320.0;
    p = p * r + 1.0 / 5040.0;
    p = p * r + 1.0 / 720.0;
    p = p * r + 1.0 / 120.0;
    p = p * r + 1.0 / 24.0;
    p = p * r + 1.0 / 6.0;
    p = p * r + 0.5;
    p = p * r + 1.0;
    p = p * r + 1.0;
    return (float) ldexp(p, (int) k);
}

// erf(x) as a fixed sequence of IEEE double operations rounded once to f32:
// for |x| < 4, x p(u) with u = x^2 / 8 - 1 and p the degree-26 Chebyshev
// interpolant of erf(sqrt t) / sqrt t on t in [0, 16] (t = 8 (u + 1)), in
// powers of u by Horner's rule with fused multiply-adds; +-1 beyond, where the
// exact value rounds to +-1 in f32. p is within 2.1e-16 of the function
// relative, and the sum is well conditioned (the |terms| add up to 1.13), so
// the f32 result is the rounded exact value but for values within ~5e-16 of a
// rounding boundary. The CPU reference sums the 64 Maclaurin terms in double
// (126 operations; ~1e-10 absolute near |x| = 4 by cancellation): over 4.5
// million f32 values the two differ in none below |x| = 3 and in 41 above it,
// the reference being the misrounded one in each.
// A value costs 28 double operations instead of 128, which bound the epilogues
// of the encoder's GELU products (the first convolution's column GEMM, 46
// million GELUs: 270 -> 161 us).
static constexpr double kErfCoef[27] = {
    0x1.6a040781a499cp-2, -0x1.69a0ccda3df7bp-3, 0x1.0dabaf0613e39p-3, -0x1.b92e95c190710p-4,
    0x1.717efc7844a6cp-4, -0x1.3215d8b7af3c1p-4, 0x1.ea97f14b7dc46p-5, -0x1.76e8648e205dbp-5,
    0x1.0ed52bfffd118p-5, -0x1.7034fab7f107ep-6, 0x1.d63529bec8d80p-7, -0x1.1a0231cf18493p-7,
    0x1.3e150dd441188p-8, -0x1.51ef24c69b64ep-9, 0x1.52d9f537fb997p-10, -0x1.4158cdbca87c1p-11,
    0x1.20eb1d497b902p-12, -0x1.edfa4cf86b66ap-14, 0x1.917dba92dfc16p-15, -0x1.34f439f8220f0p-16,
    0x1.cad408e75faaap-18, -0x1.5648b45cedfc6p-19, 0x1.cd204a8e02514p-21, -0x1.c13100c22049cp-23,
    0x1.26ea8a0fd734fp-24, -0x1.7f1f9da9b2298p-25, 0x1.af4c0b060735bp-27,
};

__device__ __forceinline__ float erff_det(float x) {
    if (x != x) return x;
    const double xd = (double) x;
    if (xd >= 4.0) return 1.0f;
    if (xd <= -4.0) return -1.0f;
    const double u = __builtin_fma(xd * xd, 0.125, -1.0);
    double p = kErfCoef[26];
#pragma unroll
    for (int n = 25; n >= 0; n--) p = __builtin_fma(p, u, kErfCoef[n]);
    return (float) (xd * p);
}

// GELU_ERF (ggml_vec_gelu_erf_f32): 0.5 x (1 + erf(x / sqrt 2)) in f32
__device__ __forceinline__ float gelu_erf_det(float x) { return 0.5f * x * (1.0f + erff_det(x * 0.70710678118654752440f)); }

// gelu_erf_det of NV values at once: the same operations per value (so the
// same bits), the NV Horner chains interleaved step by step so that a lane
// has NV independent double operations in flight instead of one chain; the
// series is evaluated for every value and the NaN / |x| >= 4 cases selected
// after it (their series result is discarded)
template <int NV>
__device__ __forceinline__ void gelu_erf_det_n(float (&x)[NV]) {
    double xd[NV], u[NV], p[NV];
#pragma unroll
    for (int e = 0; e < NV; e++) {
        xd[e] = (double) (x[e] * 0.70710678118654752440f);
        u[e] = __builtin_fma(xd[e] * xd[e], 0.125, -1.0);
        p[e] = kErfCoef[26];
    }
#pragma unroll
    for (int n = 25; n >= 0; n--)
#pragma unroll
        for (int e = 0; e < NV; e++) p[e] = __builtin_fma(p[e], u[e], kErfCoef[n]);
#pragma unroll
    for (int e = 0; e < NV; e++) {
        const float a = x[e] * 0.70710678118654752440f;
        float er = (float) (xd[e] * p[e]);
        if (xd[e] >= 4.0) er = 1.0f;
        if (xd[e] <= -4.0) er = -1.0f;
        if (a != a) er = a;
        x[e] = 0.5f * x[e] * (1.0f + er);
    }
}

__device__ __forceinline__ void sincosf_det(float x, float & s_out, float & c_out) {
    const double xd = (double) x;
    const double k = rint(xd * 0.63661977236758134308);
    const double r = (xd - k * 1.5707963267341256458) - k * 6.0771005065061922341e-11;
    const double r2 = r * r;
    double s = -1.0 / 355687428096000.0;
    s = s * r2 + 1.0 / 1307674368000.0;
    s = s * r2 - 1.0 / 6227020800.0;
    s = s * r2 + 1.0 / 39916800.0;
    s = s * r2 - 1.0 / 362880.0;
    s = s * r2 + 1.0 / 5040.0;
    s = s * r2 - 1.0 / 120.0;
    s = s * r2 + 1.0 / 6.0;
    s = r - (r * r2) * s;
    double c = 1.0 / 6402373705728000.0;
    c = c * r2 - 1.0 / 20922789888000.0;
    c = c * r2 + 1.0 / 87178291200.0;
    c = c * r2 - 1.0 / 479001600.0;
    c = c * r2 + 1.0 / 3628800.0;
    c = c * r2 - 1.0 / 40320.0;
    c = c * r2 + 1.0 / 720.0;
    c = c * r2 - 1.0 / 24.0;
    c = c * r2 + 0.5;
    c = 1.0 - r2 * c;
    const int q = (int) (((long long) k) & 3);
    double so, co;
    if (q == 0) {
        so = s;
        co = c;
    } else if (q == 1) {
        so = c;
        co = -s;
    } else if (q == 2) {
        so = -s;
        co = -c;
    } else {
        so = -c;
        co = s;
    }
    s_out = (float) so;
    c_out = (float) co;
}

}  // namespace mi355x
