// rb_philox.hh -- device-side counter-based random streams for gfx950.
//
// Philox4x32-10 (the RandBLAS DefaultRNG, RandBLAS/base.hh:53) and the maps
// RandBLAS applies to its words: uneg11 / u01 and the Box-Muller transform
// (RandBLAS/random_gen.hh:60-137, Random123 uniform.hpp / boxmuller.hpp).
//
// Box-Muller needs sin, cos and log of float arguments.  Their values are
// defined by the oracle's series (Taylor / atanh in double precision, one
// final rounding to float); here the same floats are reached with less work:
//   sin/cos(t): t = PIf u reduced by k pi/2 (k = rint(2u), one fma: k pi/2 -
//     t loses nothing that the final rounding sees), minimax polynomials of
//     six coefficients in r^2 (relative errors 2^-58 and 2^-54);
//   log(u): u = 2^e m, m in [1/sqrt2, sqrt2), log m = 2 atanh(s), s =
//     f / (2 + f), f = m - 1: the quotient from v_rcp_f32 and one cubic
//     Newton step (2^-52), six minimax coefficients in s^2 (2^-52).
// The resulting floats equal the series' for every one of the 2^32 words that
// either factor can be given (checked exhaustively, on the CPU with the
// reciprocal seed off by -1, 0 and +1 ulp, and on gfx950), so the operators'
// entries are the same bits as the oracle's.  Every step is an IEEE operation
// with an explicit fma where fused, and the library is compiled with
// -ffp-contract=off, so results do not depend on the compiler's contraction
// choices.
//
// Cost, measured issue cycles per wave and SIMD on gfx950: f64 fma / mul /
// add, 32-bit integer multiplies and f32 <-> f64 conversions 4, f32 and
// logic operations 2, v_rcp / v_rsq / v_sqrt_f32 8, v_rcp_f64 16; FP64 and
// FP32 MFMAs share these issue cycles (they do not overlap with VALU work),
// BF16 ones do not.  fill_dense of 4096 x 65536 FP32 Gaussians, which is this
// generator and one store: 365 us = 7.3e11 entries/s (508 us with the series
// themselves: degree 16-17 sin / cos, an IEEE division, sqrtf and two-input
// xors in Philox).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rbx {

constexpr uint32_t PH_M0 = 0xD2511F53u;
constexpr uint32_t PH_M1 = 0xCD9E8D57u;
constexpr uint32_t PH_W0 = 0x9E3779B9u;
constexpr uint32_t PH_W1 = 0xBB67AE85u;

// 128-bit counter held as two 64-bit halves (word 0 = low 32 bits of lo).
struct Ctr128 {
    uint64_t lo, hi;
};

__host__ __device__ inline Ctr128 ctr_from_words(const uint32_t c[4]) {
    return Ctr128{(uint64_t)c[0] | ((uint64_t)c[1] << 32), (uint64_t)c[2] | ((uint64_t)c[3] << 32)};
}

__host__ __device__ inline Ctr128 ctr_add(Ctr128 c, uint64_t n) {
    uint64_t lo = c.lo + n;
    return Ctr128{lo, c.hi + (lo < n ? 1u : 0u)};
}

__host__ __device__ inline void ctr_to_words(Ctr128 c, uint32_t w[4]) {
    w[0] = (uint32_t)c.lo;
    w[1] = (uint32_t)(c.lo >> 32);
    w[2] = (uint32_t)c.hi;
    w[3] = (uint32_t)(c.hi >> 32);
}

__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}

// Philox4x32-10 on one counter.  The key words are wave-uniform in every
// caller, so the Weyl bumps stay on the scalar unit.
__device__ __forceinline__ uint4 philox4x32_10(Ctr128 c, uint32_t k0, uint32_t k1) {
    uint32_t x0 = (uint32_t)c.lo, x1 = (uint32_t)(c.lo >> 32);
    uint32_t x2 = (uint32_t)c.hi, x3 = (uint32_t)(c.hi >> 32);
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r > 0) {
            k0 += PH_W0;
            k1 += PH_W1;
        }
        uint64_t p0 = (uint64_t)PH_M0 * x0;
        uint64_t p1 = (uint64_t)PH_M1 * x2;
        uint32_t y0 = xor3((uint32_t)(p1 >> 32), x1, k0);
        uint32_t y2 = xor3((uint32_t)(p0 >> 32), x3, k1);
        x1 = (uint32_t)p1;
        x3 = (uint32_t)p0;
        x0 = y0;
        x2 = y2;
    }
    return make_uint4(x0, x1, x2, x3);
}

// (float)(int32)w * 2^-31 + 2^-32; the product is exact, so one fma.
__device__ __forceinline__ float uneg11(uint32_t w) { return __fmaf_rn((float)(int32_t)w, 0x1p-31f, 0x1p-32f); }
// (float)w * 2^-32 + 2^-33
__device__ __forceinline__ float u01(uint32_t w) { return __fmaf_rn((float)w, 0x1p-32f, 0x1p-33f); }

// sin and cos of PIf * uneg11(w) (the float product): the angle factors of a
// Box-Muller draw.
__device__ __forceinline__ void bm_sincos(uint32_t w, float &s_out, float &c_out) {
    const float u = uneg11(w);
    const double t = (double)__fmul_rn(3.1415926535897932f, u);
    // k = rint(2u) with the quadrant k mod 4 in the sum's low bits
    const float km = __fmaf_rn(2.0f, u, 0x1.8p23f);
    const uint32_t q = __float_as_uint(km);
    const double r = __fma_rn((double)__fsub_rn(0x1.8p23f, km), 0x1.921fb54442d18p+0, t);
    const double r2 = __dmul_rn(r, r);
    double ps = 0x1.5d932ee04e218p-33;
    ps = __fma_rn(ps, r2, -0x1.ae5e66d38ca7bp-26);
    ps = __fma_rn(ps, r2, 0x1.71de357872c1dp-19);
    ps = __fma_rn(ps, r2, -0x1.a01a019c12695p-13);
    ps = __fma_rn(ps, r2, 0x1.111111110f880p-7);
    ps = __fma_rn(ps, r2, -0x1.5555555555549p-3);
    const float sv = (float)__fma_rn(__dmul_rn(r, r2), ps, r);
    double pc = 0x1.1b95fd680bb2cp-29;
    pc = __fma_rn(pc, r2, -0x1.27df6c029fc1ep-22);
    pc = __fma_rn(pc, r2, 0x1.a019f8841065cp-16);
    pc = __fma_rn(pc, r2, -0x1.6c16c1648a8e4p-10);
    pc = __fma_rn(pc, r2, 0x1.555555554f951p-5);
    pc = __fma_rn(pc, r2, -0x1.fffffffffffa3p-2);
    const float cv = (float)__fma_rn(r2, pc, 1.0);
    const bool odd = (q & 1) != 0;
    // quadrants 2, 3 negate the sine, 1, 2 the cosine
    s_out = __uint_as_float(__float_as_uint(odd ? cv : sv) ^ ((q << 30) & 0x80000000u));
    c_out = __uint_as_float(__float_as_uint(odd ? sv : cv) ^ (((q + 1) << 30) & 0x80000000u));
}

// sqrtf(-2 logf(u01(w))), the radius factor.
__device__ __forceinline__ float bm_radius(uint32_t w) {
    const uint32_t b = __float_as_uint(u01(w)) - 0x3f3504f3u;  // from 1/sqrt2
    const float m = __uint_as_float((b & 0x7fffffu) + 0x3f3504f3u);
    const float ff = __fsub_rn(m, 1.0f);  // exact
    const double f = (double)ff, d = __dadd_rn(f, 2.0);
    double y = (double)__builtin_amdgcn_rcpf(__fadd_rn(ff, 2.0f));
    const double e1 = __fma_rn(-d, y, 1.0);
    y = __fma_rn(y, __fma_rn(e1, e1, e1), y);
    const double s = __dmul_rn(f, y), s2 = __dmul_rn(s, s);
    double p = 0x1.58786ae4b778cp-3;
    p = __fma_rn(p, s2, 0x1.732c1304abcfep-3);
    p = __fma_rn(p, s2, 0x1.c72278a03a957p-3);
    p = __fma_rn(p, s2, 0x1.24924176cc058p-2);
    p = __fma_rn(p, s2, 0x1.999999a294cb3p-2);
    p = __fma_rn(p, s2, 0x1.5555555553960p-1);
    const double lm = __fma_rn(__dmul_rn(s, s2), p, __dadd_rn(s, s));
    const float x = __fmul_rn(-2.0f, (float)__fma_rn((double)((int32_t)b >> 23), 0x1.62e42fefa39efp-1, lm));
    // correctly rounded square root of x in {-0} U [2^-23, 46): one Newton
    // correction of x rsq(x), with the residual exact in the fma
    const float q = __builtin_amdgcn_rsqf(fmaxf(x, 0x1p-100f));
    const float r = __fmul_rn(x, q);
    return __fmaf_rn(__fmaf_rn(-r, r, x), __fmul_rn(0.5f, q), r);
}

// r123::boxmuller(u0, u1): (r*sin(pi_f*uneg11(u0)), r*cos(...)), r = sqrtf(-2 logf(u01(u1))).
__device__ __forceinline__ float2 boxmuller(uint32_t w0, uint32_t w1) {
    float s, c;
    bm_sincos(w0, s, c);
    const float r = bm_radius(w1);
    return make_float2(__fmul_rn(s, r), __fmul_rn(c, r));
}

// One Philox call -> four operator entries (random_gen.hh:85-137).
__device__ __forceinline__ float4 gen4(bool gauss, Ctr128 c, uint32_t k0, uint32_t k1) {
    uint4 w = philox4x32_10(c, k0, k1);
    if (gauss) {
        float2 a = boxmuller(w.x, w.y);
        float2 b = boxmuller(w.z, w.w);
        return make_float4(a.x, a.y, b.x, b.y);
    }
    return make_float4(uneg11(w.x), uneg11(w.y), uneg11(w.z), uneg11(w.w));
}

// gen4 with the two Box-Muller pairs kept apart by scheduling fences, for
// kernels whose register budget cannot hold both pairs' temporaries at once.
__device__ __forceinline__ float4 gen4_lean(bool gauss, Ctr128 c, uint32_t k0, uint32_t k1) {
    uint4 w = philox4x32_10(c, k0, k1);
    if (gauss) {
        __builtin_amdgcn_sched_barrier(0);
        float2 a = boxmuller(w.x, w.y);
        __builtin_amdgcn_sched_barrier(0);
        float2 b = boxmuller(w.z, w.w);
        __builtin_amdgcn_sched_barrier(0);
        return make_float4(a.x, a.y, b.x, b.y);
    }
    return make_float4(uneg11(w.x), uneg11(w.y), uneg11(w.z), uneg11(w.w));
}

__device__ __forceinline__ float f4_get(const float4 &v, int t) {
    return t == 0 ? v.x : (t == 1 ? v.y : (t == 2 ? v.z : v.w));
}

// Entry value in precision T: Gaussians are promoted; uniforms are promoted
// and then scaled by (T)sqrt(3) as in dense_skops.hh:587-590.
template <typename T>
__device__ __forceinline__ T entry_value(float v, bool gauss);
template <>
__device__ __forceinline__ double entry_value<double>(float v, bool gauss) {
    return gauss ? (double)v : __dmul_rn((double)v, 0x1.bb67ae8584caap+0);
}
template <>
__device__ __forceinline__ float entry_value<float>(float v, bool gauss) {
    return gauss ? v : __fmul_rn(v, 0x1.bb67aep+0f);  // (float)sqrt(3.0)
}

// The factor of entry_value: (T)v * entry_scale<T>(gauss) are the same bits.
template <typename T>
__host__ __device__ constexpr T entry_scale(bool gauss) {
    return gauss ? (T)1 : (sizeof(T) == 8 ? (T)0x1.bb67ae8584caap+0 : (T)0x1.bb67aep+0f);
}

// bfloat16 (as its 16 bits) nearest to x, ties to even; x not NaN.
__host__ __device__ __forceinline__ uint16_t bf16_rne(float x) {
#ifdef __HIP_DEVICE_COMPILE__
    uint32_t u = __float_as_uint(x);
#else
    uint32_t u;
    __builtin_memcpy(&u, &x, 4);
#endif
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// Operator entry of the BF16 operator: the FP32 entry rounded to bfloat16.
template <>
__device__ __forceinline__ uint16_t entry_value<uint16_t>(float v, bool gauss) {
    return bf16_rne(entry_value<float>(v, gauss));
}

}  // namespace rbx
