// rbx_chain.hh -- sequential floating-point summation of non-negative terms
// as integer arithmetic, so that it can be done in parallel with the same
// bits as the loop  s = s + w[0]; s = s + w[1]; ...
//
// While the running sum stays in one binade (exponent field e, spacing u),
// s is an integer multiple of u and so is every rounded sum: RN(s + w) =
// s + r u with r = w / u rounded to an integer, a function of w and e alone
// unless w / u lies exactly half way between two integers, where ties-to-even
// makes it depend on the parity of s / u as well.  The sum's bit pattern,
// read as an integer, advances by r.  A run of terms is therefore a pair of
// advances, one for each parity of the sum it starts from; pairs compose
// associatively (a scan), and the sum leaves the binade exactly at the first
// term whose advance reaches the next exponent: that one term is added in
// floating point, and the scan goes on with the new exponent.
// Advances are capped at one whole binade's length, which is enough to leave it.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

namespace rbx {

template <typename T>
struct ChainFp;
template <>
struct ChainFp<double> {
    static constexpr int MANT = 52, EXP_INF = 2047;
};
template <>
struct ChainFp<float> {
    static constexpr int MANT = 23, EXP_INF = 255;
};

// bit pattern of a non-negative value (or -0, taken as 0) as an integer, and back
__host__ __device__ inline int64_t chain_bits(double s) {
    int64_t b;
    memcpy(&b, &s, 8);
    return b & 0x7fffffffffffffffll;
}
__host__ __device__ inline int64_t chain_bits(float s) {
    uint32_t b;
    memcpy(&b, &s, 4);
    return (int64_t)(b & 0x7fffffffu);
}
template <typename T>
__host__ __device__ inline T chain_value(int64_t bits);
template <>
__host__ __device__ inline double chain_value<double>(int64_t bits) {
    double s;
    memcpy(&s, &bits, 8);
    return s;
}
template <>
__host__ __device__ inline float chain_value<float>(int64_t bits) {
    const uint32_t b = (uint32_t)bits;
    float s;
    memcpy(&s, &b, 4);
    return s;
}

template <typename T>
__host__ __device__ inline constexpr int64_t chain_cap() {
    return 2ll << ChainFp<T>::MANT;
}
// exponent field of a sum; subnormals share the spacing of field 1
template <typename T>
__host__ __device__ inline int chain_exp(int64_t bits) {
    const int e = (int)(bits >> ChainFp<T>::MANT);
    return e > 1 ? e : 1;
}
// first bit pattern past the binade of exponent field e
template <typename T>
__host__ __device__ inline uint64_t chain_limit(int e) {
    return (uint64_t)(e + 1) << ChainFp<T>::MANT;
}

// advance of the sum's bits over a run of terms, for a sum of even (d0) or
// odd (d1) bits at its start
struct Advance {
    int64_t d0, d1;
};

template <typename T>
__host__ __device__ inline Advance chain_compose(Advance a, Advance b) {
    const int64_t cap = chain_cap<T>();
    int64_t d0 = a.d0 + ((a.d0 & 1) ? b.d1 : b.d0);
    int64_t d1 = a.d1 + ((a.d1 & 1) ? b.d0 : b.d1);
    d0 = d0 < cap ? d0 : cap;
    d1 = d1 < cap ? d1 : cap;
    return Advance{d0, d1};
}

// one term w >= 0 onto a sum of exponent field e; an infinite sum stays
template <typename T>
__host__ __device__ inline Advance chain_term(T w, int e) {
    constexpr int MANT = ChainFp<T>::MANT;
    if (e >= ChainFp<T>::EXP_INF) return Advance{0, 0};
    const int64_t b = chain_bits(w);
    const int ew = chain_exp<T>(b);
    const int sh = e - ew;
    if (sh < 0) return Advance{chain_cap<T>(), chain_cap<T>()};
    if (sh > MANT + 1) return Advance{0, 0};
    const int64_t m = b - ((int64_t)(ew - 1) << MANT);  // significand
    const int64_t q = m >> sh, rem2 = (m - (q << sh)) * 2, one = 1ll << sh;
    if (rem2 == one && sh > 0) return Advance{q + (q & 1), q + ((q + 1) & 1)};
    const int64_t r = q + (rem2 > one ? 1 : 0);
    return Advance{r, r};
}

}  // namespace rbx
