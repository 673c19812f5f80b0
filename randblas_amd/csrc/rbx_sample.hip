// rbx_sample.hip -- index sampling and CDF preparation on the device:
//   sample_indices_iid_uniform  (RandBLAS/util.hh:516-560)
//   sample_indices_iid          (RandBLAS/util.hh:493-514)
//   weights_to_cdf              (RandBLAS/util.hh:459-472)
// Each sample reads the same Philox words as the reference's sequential loop:
// without signs, sample i uses word i mod 4 of counter ctr + floor(i / 4);
// with Rademacher signs, sample i uses words 2(i mod 2), 2(i mod 2) + 1 of
// counter ctr + floor(i / 2).  The returned state is the seed advanced by the
// number of counters the loop touched.  One thread per counter.
#include <algorithm>
#include <cmath>
#include <limits>
#include <type_traits>
#include <vector>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "rbx_internal.hh"
#include "rbx_chain.hh"

namespace rbx {

// (sint) ((double) n * ((double) uneg11(w) + 1) / 2), util.hh:531-533
__device__ __forceinline__ int64_t uniform_index(uint32_t w, double dN) {
    const double u = __dmul_rn(__dadd_rn((double)uneg11(w), 1.0), 0.5);
    return (int64_t)__dmul_rn(dN, u);
}

template <typename T>
__global__ __launch_bounds__(256) void iid_uniform_kernel(Ctr128 ctr, uint32_t k0, uint32_t k1, int64_t n, int64_t k,
                                                          int64_t *samples, T *rademachers) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int per = rademachers ? 2 : 4;
    const int64_t i0 = c * per;
    if (i0 >= k) return;
    const uint4 w4 = philox4x32_10(ctr_add(ctr, (uint64_t)c), k0, k1);
    const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
    const double dN = (double)n;
    // whole counters with 16-byte aligned outputs: vector stores (a thread's
    // samples are contiguous, so its 32 or 16 bytes go out in one or two pieces)
    const bool vec = i0 + per <= k && ((uintptr_t)(samples + i0) & 15) == 0 &&
                     (rademachers == nullptr || ((uintptr_t)(rademachers + i0) & (2 * sizeof(T) - 1)) == 0);
    if (vec) {
        typedef long long i64x2 __attribute__((ext_vector_type(2)));
        typedef T tx2 __attribute__((ext_vector_type(2)));
        if (rademachers) {
            const i64x2 sv = {uniform_index(w[0], dN), uniform_index(w[2], dN)};
            const tx2 rv = {uneg11(w[1]) >= 0.0f ? (T)1 : (T)-1, uneg11(w[3]) >= 0.0f ? (T)1 : (T)-1};
            *(i64x2 *)(samples + i0) = sv;
            *(tx2 *)(rademachers + i0) = rv;
        } else {
            const i64x2 s01 = {uniform_index(w[0], dN), uniform_index(w[1], dN)};
            const i64x2 s23 = {uniform_index(w[2], dN), uniform_index(w[3], dN)};
            *(i64x2 *)(samples + i0) = s01;
            *(i64x2 *)(samples + i0 + 2) = s23;
        }
        return;
    }
    for (int q = 0; q < per && i0 + q < k; ++q) {
        if (rademachers) {
            samples[i0 + q] = uniform_index(w[2 * q], dN);
            rademachers[i0 + q] = uneg11(w[2 * q + 1]) >= 0.0f ? (T)1 : (T)-1;
        } else {
            samples[i0 + q] = uniform_index(w[q], dN);
        }
    }
}

// u = ((T) uneg11(w) + 1) / 2 in T (uneg11_to_u01<T>, util.hh:474-477), then
// the first index whose CDF value is not below u, by std::lower_bound's own
// probe sequence (half = len / 2, mid = lo + half).  The first CDF_LEVELS
// levels of that sequence probe at most 2^CDF_LEVELS - 1 positions, the
// same for every u: each workgroup loads them into LDS as a heap-ordered
// tree (node t, children 2t for cdf[mid] >= u and 2t + 1 for cdf[mid] < u),
// so only the remaining levels read global memory; results are identical
// to the plain search for any array.  The grid is a few workgroups per CU,
// each looping over counters, so a tree serves many draws; a thread's four
// searches of a counter run in lockstep, their global probes in flight
// together.
constexpr int CDF_LEVELS = 12, CDF_NODES = (1 << CDF_LEVELS) - 1;
template <typename T>
__global__ __launch_bounds__(256) void iid_cdf_kernel(Ctr128 ctr, uint32_t k0, uint32_t k1, int64_t n, const T *cdf,
                                                      int64_t k, int64_t *samples) {
    __shared__ T tree[CDF_NODES + 1];
    for (int t = threadIdx.x + 1; t <= CDF_NODES; t += blockDim.x) {
        int64_t lo = 0, len = n;
        const int depth = 31 - __builtin_clz((unsigned)t);
        for (int bit = depth - 1; bit >= 0; --bit) {
            const int64_t half = len / 2, mid = lo + half;
            if ((t >> bit) & 1) {
                lo = mid + 1;
                len -= half + 1;
            } else {
                len = half;
            }
        }
        tree[t] = len > 0 ? cdf[lo + len / 2] : (T)0;  // unused when len == 0
    }
    __syncthreads();
    const int64_t ncounters = (k + 3) / 4;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < ncounters;
         c += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i0 = c * 4;
        const uint4 w4 = philox4x32_10(ctr_add(ctr, (uint64_t)c), k0, k1);
        const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
        T u[4];
        int64_t lo[4], len[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            u[q] = ((T)uneg11(w[q]) + (T)1) / (T)2;
            lo[q] = 0;
            len[q] = n;
            int t = 1;
            for (int lev = 0; lev < CDF_LEVELS && len[q] > 0; ++lev) {
                const int64_t half = len[q] / 2;
                if (tree[t] < u[q]) {
                    lo[q] += half + 1;
                    len[q] -= half + 1;
                    t = 2 * t + 1;
                } else {
                    len[q] = half;
                    t = 2 * t;
                }
            }
        }
        bool more = true;
        while (more) {
            more = false;
            T v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = len[q] > 0 ? cdf[lo[q] + len[q] / 2] : (T)0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (len[q] > 0) {
                    const int64_t half = len[q] / 2;
                    if (v[q] < u[q]) {
                        lo[q] += half + 1;
                        len[q] -= half + 1;
                    } else {
                        len[q] = half;
                    }
                    more |= len[q] > 0;
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (i0 + q < k) samples[i0 + q] = lo[q];
    }
}

// Many draws from one array: the search by a table made in the same call.
// key(x) = floor(2^31 x), clamped to [0, 2^31), is monotone; its high bits pick
// one of NB buckets of [0, 1), its low 16 order the entries inside one.
//   start[b]  the first index whose key is in bucket b or later (a copy in LDS)
//   low[i]    the low 16 bits of cdf[i]'s key: a quarter of the array's bytes
// A draw searches low[] inside its bucket; only where the keys agree in all 31
// bits does it go on in cdf[] itself, so the index is lower_bound's.  That
// needs an ascending array: cdf_table_kernel looks, and a draw from any other
// runs the plain probe sequence.  Long arrays (NEAR) have many entries to a
// bucket, and one 16-byte load around the place that even spacing would give
// mostly ends the search.  Bound by these loads' addresses (one lane a clock)
// and the L2s: 2^24 draws from 10^6 FP64 weights 178 us, 0.75 TB/s of indices
// written; 349 us without that load, 879 us by the probe tree below, whose last
// eight levels read 8 MB that no XCD's L2 holds.
template <typename T>
__device__ __forceinline__ uint32_t cdf_key(T x) {
    return (uint32_t)fmin(fmax((double)x * 0x1p31, 0.0), 0x1.fffffffcp30);
}
constexpr int64_t CDF_TABLE_BLOCKS = 1024;
constexpr int CDF_BUCKET_BITS = 15, CDF_BUCKETS = 1 << CDF_BUCKET_BITS, CDF_LOW_BITS = 31 - CDF_BUCKET_BITS;
static_assert(CDF_LOW_BITS <= 16, "16-bit keys inside a bucket");

template <typename T>
__global__ __launch_bounds__(256) void cdf_table_kernel(int64_t n, const T *cdf, uint32_t *start, uint16_t *low,
                                                        int *unsorted) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    bool bad = false;
    for (int64_t i = g; i < n; i += stride) {
        const T x = cdf[i], y = cdf[i + 1 < n ? i + 1 : i];
        bad |= !(x <= y);
        low[i] = (uint16_t)(cdf_key(x) & ((1u << CDF_LOW_BITS) - 1));
    }
    for (int64_t b = g; b <= CDF_BUCKETS; b += stride) {
        int64_t lo = 0, len = b == CDF_BUCKETS ? 0 : n;
        if (b == CDF_BUCKETS) lo = n;
        while (len > 0) {
            const int64_t half = len / 2;
            if ((int64_t)(cdf_key(cdf[lo + half]) >> CDF_LOW_BITS) < b) {
                lo += half + 1;
                len -= half + 1;
            } else {
                len = half;
            }
        }
        start[b] = (uint32_t)lo;
    }
    const int any = __syncthreads_or(bad);
    if (threadIdx.x == 0) unsorted[blockIdx.x] = any;
}

template <typename T>
__device__ __forceinline__ int64_t cdf_lower_bound(const T *cdf, int64_t lo, int64_t len, T u) {
    while (len > 0) {
        const int64_t half = len / 2;
        if (cdf[lo + half] < u) {
            lo += half + 1;
            len -= half + 1;
        } else {
            len = half;
        }
    }
    return lo;
}

typedef uint16_t u16x8 __attribute__((ext_vector_type(8), aligned(2)));
template <typename T, bool NEAR>
__global__ __launch_bounds__(1024) void iid_cdf_table_kernel(Ctr128 ctr, uint32_t k0, uint32_t k1, int64_t n,
                                                             const T *cdf, const uint32_t *start, const uint16_t *low,
                                                             const int *unsorted, int nflags, int64_t k,
                                                             int64_t *samples) {
    __shared__ uint32_t first[CDF_BUCKETS + 1];
    for (int b = threadIdx.x; b <= CDF_BUCKETS; b += 1024) first[b] = start[b];
    int bad = 0;
    for (int b = threadIdx.x; b < nflags; b += 1024) bad |= unsorted[b];
    const bool sorted = __syncthreads_or(bad) == 0;
    const int64_t ncounters = (k + 3) / 4;
    for (int64_t c = (int64_t)blockIdx.x * 1024 + threadIdx.x; c < ncounters; c += (int64_t)gridDim.x * 1024) {
        const int64_t i0 = c * 4;
        const uint4 w4 = philox4x32_10(ctr_add(ctr, (uint64_t)c), k0, k1);
        const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
        int64_t at[4];
        if (sorted) {
            uint32_t lo[4], len[4], key[4], got[4];  // got: low[lo] where the search has seen it
            bool more = false;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t ku = cdf_key(((T)uneg11(w[q]) + (T)1) / (T)2);
                const uint32_t b = ku >> CDF_LOW_BITS;
                key[q] = ku & ((1u << CDF_LOW_BITS) - 1);
                lo[q] = first[b];
                len[q] = first[b + 1] - lo[q];
                got[q] = 1u << 16;
            }
            if constexpr (NEAR) {
                // first the eight entries around the place that even spacing would give
                u16x8 x[4];
                uint32_t at8[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t est = lo[q] + (uint32_t)(((uint64_t)len[q] * key[q]) >> CDF_LOW_BITS);
                    at8[q] = est < 4 ? 0 : (est > (uint32_t)n - 4 ? (uint32_t)n - 8 : est - 4);
                    x[q] = *(const u16x8 *)(low + at8[q]);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t end = lo[q] + len[q];
                    uint32_t a = lo[q], z = end;  // the index is in [a, z]
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const uint32_t i = at8[q] + e;
                        if (i >= lo[q] && i < end) {
                            if (x[q][e] < key[q]) {
                                a = i + 1;
                            } else if (i < z) {
                                z = i;
                                got[q] = x[q][e];
                            }
                        }
                    }
                    lo[q] = a;
                    len[q] = z - a;
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) more |= len[q] > 0;
            while (more) {
                more = false;
                uint32_t v[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = len[q] > 0 ? low[lo[q] + len[q] / 2] : 0u;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (len[q] > 0) {
                        const uint32_t half = len[q] / 2;
                        if (v[q] < key[q]) {
                            lo[q] += half + 1;
                            len[q] -= half + 1;
                        } else {
                            got[q] = v[q];
                            len[q] = half;
                        }
                        more |= len[q] > 0;
                    }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                at[q] = lo[q];
                if (got[q] == key[q]) {
                    const T u = ((T)uneg11(w[q]) + (T)1) / (T)2;
                    at[q] = cdf_lower_bound(cdf, at[q], first[(cdf_key(u) >> CDF_LOW_BITS) + 1] - at[q], u);
                }
            }
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) at[q] = cdf_lower_bound(cdf, 0, n, ((T)uneg11(w[q]) + (T)1) / (T)2);
        }
        typedef long long i64x2 __attribute__((ext_vector_type(2), aligned(8)));
        if (i0 + 4 <= k) {
            *(i64x2 *)(samples + i0) = i64x2{at[0], at[1]};
            *(i64x2 *)(samples + i0 + 2) = i64x2{at[2], at[3]};
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (i0 + q < k) samples[i0 + q] = at[q];
        }
    }
}

// weights_to_cdf: the prefix sums in the reference's order, with the bits of
// its loop  sum = sum + max(w[i], 0).  The loop is one dependent addition per
// weight (10.4 ms for 10^6 FP64 weights on one thread, 10 ns an addition);
// inside a binade of the sum it is integer arithmetic that scans in parallel
// (rbx_chain.hh), so the work is five short kernels over blocks of CDF_BLK:
//   cdf_sums_kernel     block sums in FP64, in any order (a guess only), and
//                       the first weight below error_if_below
//   cdf_guess_kernel    their prefix sums: the binade each block is in
//   cdf_advance_kernel  each block's advance in its guessed binade
//   cdf_chain_kernel    one workgroup composes the blocks' advances in order,
//                       64 at a time, as long as the exact sum is in the
//                       guessed binade and stays there; a block that fails
//                       the test (a binade is left inside it, or the guess
//                       was wrong) is summed term by term in integer scans
//                       with the exact exponent, one more for every binade
//                       left.  No result depends on the guesses.
//   cdf_write_kernel    each block's partial sums from its exact start, scaled
// 10^6 FP64 weights: 9 blocks leave a binade.  Bound by latency: the chain
// kernel's dependent scans (157 us of them; 135 with the first CDF_HEAD terms
// added one by one; 3122 weights and as many draws 106 -> 79 us).  Arrays of a few blocks skip the first three.
// Meta: status 0 ok (inv = 1 / sum); 1 + i: w[i] < error_if_below (w[0..i)
// hold the partial sums, as when the reference throws there); -1: the total
// is below sqrt(n) * eps (w holds the partial sums, unscaled).
constexpr int CDF_BLK = 2048, CDF_PER = CDF_BLK / 256;
constexpr int CDF_HEAD = 192;  // terms (2 us) whose sums may leave eight binades (3 us each in scans)
constexpr int64_t CDF_DIRECT = 4;  // blocks that the chain kernel takes by itself
struct CdfMeta {
    long long status, first;  // first: weights before the first refused one
    double inv;
};

template <typename T>
__global__ __launch_bounds__(256) void cdf_sums_kernel(int64_t n, const T *w, T error_if_below, double *bsum,
                                                       int *bbad) {
    __shared__ double red[4];
    __shared__ int bad_sh;
    const int tid = threadIdx.x;
    const int64_t i0 = (int64_t)blockIdx.x * CDF_BLK;
    if (tid == 0) bad_sh = CDF_BLK;
    __syncthreads();
    double v = 0.0;
#pragma unroll
    for (int q = 0; q < CDF_PER; ++q) {
        const int e = tid + 256 * q;
        if (i0 + e < n) {
            const T x = w[i0 + e];
            if (!(x >= error_if_below)) atomicMin(&bad_sh, e);
            v += x > (T)0 ? (double)x : 0.0;
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
    if ((tid & 63) == 0) red[tid >> 6] = v;
    __syncthreads();
    if (tid == 0) {
        bsum[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
        bbad[blockIdx.x] = bad_sh;
    }
}

// bsum[0 .. nb) -> exclusive prefix sums in bsum[0 .. nb]; first refused weight
__global__ __launch_bounds__(1024) void cdf_guess_kernel(int64_t n, int64_t nb, double *bsum, const int *bbad,
                                                         CdfMeta *meta) {
    __shared__ double wsum[16];
    __shared__ unsigned long long first_sh;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) first_sh = (unsigned long long)n;
    __syncthreads();
    double carry = 0.0;
    for (int64_t b0 = 0; b0 < nb; b0 += 1024) {
        const int64_t b = b0 + tid;
        const double x = b < nb ? bsum[b] : 0.0;
        if (b < nb && bbad[b] < CDF_BLK)
            atomicMin(&first_sh, (unsigned long long)(b * CDF_BLK + bbad[b]));
        double v = x;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double y = __shfl_up(v, off);
            if (lane >= off) v += y;
        }
        if (lane == 63) wsum[wave] = v;
        __syncthreads();
        double pre = carry, tot = carry;
        for (int q = 0; q < 16; ++q) {
            if (q < wave) pre += wsum[q];
            tot += wsum[q];
        }
        if (b < nb) bsum[b] = pre + (v - x);
        carry = tot;
        __syncthreads();
    }
    if (tid == 0) {
        bsum[nb] = carry;
        meta->first = (long long)first_sh;
    }
}

template <typename T>
__device__ __forceinline__ Advance shfl_up_advance(Advance a, int off) {
    return Advance{(int64_t)__shfl_up((long long)a.d0, off), (int64_t)__shfl_up((long long)a.d1, off)};
}
// inclusive scan of the lanes' advances
template <typename T>
__device__ __forceinline__ Advance wave_scan_advance(Advance a, int lane) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const Advance p = shfl_up_advance<T>(a, off);
        if (lane >= off) a = chain_compose<T>(p, a);
    }
    return a;
}

// A block's weights from memory into LDS, negative ones (not below the bound) as 0.
template <typename T>
__device__ __forceinline__ void cdf_load_block(const T *w, int len, T *wbuf, int tid) {
#pragma unroll
    for (int q = 0; q < CDF_PER; ++q) {
        const int e = tid + 256 * q;
        if (e < len) {
            const T x = w[e];
            wbuf[e] = x < (T)0 ? (T)0 : x;
        }
    }
}

template <typename T>
__global__ __launch_bounds__(256) void cdf_advance_kernel(const T *w, const double *prefix, const CdfMeta *meta,
                                                          Advance *adv, int *bexp) {
    __shared__ T wbuf[CDF_BLK];
    __shared__ Advance wtot[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t b = blockIdx.x, i0 = b * CDF_BLK;
    const int64_t left = meta->first - i0;
    const int len = left <= 0 ? 0 : (left < CDF_BLK ? (int)left : CDF_BLK);
    const int e = chain_exp<T>(chain_bits((T)prefix[b]));
    if (e != chain_exp<T>(chain_bits((T)prefix[b + 1]))) {  // leaves its binade: the chain kernel's work
        if (tid == 0) bexp[b] = -1;
        return;
    }
    cdf_load_block(w + i0, len, wbuf, tid);
    __syncthreads();
    Advance a{0, 0};
#pragma unroll
    for (int q = 0; q < CDF_PER; ++q) {
        const int i = CDF_PER * tid + q;
        if (i < len) a = chain_compose<T>(a, chain_term<T>(wbuf[i], e));
    }
    a = wave_scan_advance<T>(a, lane);
    if (lane == 63) wtot[wave] = a;
    __syncthreads();
    if (tid == 0) {
        a = wtot[0];
#pragma unroll
        for (int q = 1; q < 4; ++q) a = chain_compose<T>(a, wtot[q]);
        adv[b] = a;
        bexp[b] = e;
    }
}

// start[b]: the bits of the sum before block b, or -1 when this kernel has
// written the block's partial sums itself.  adv == nullptr: every block is
// summed here, and the refused weight looked for here.
template <typename T>
__global__ __launch_bounds__(256) void cdf_chain_kernel(int64_t n, T *w, T error_if_below, int64_t nb,
                                                        const Advance *adv, const int *bexp, int64_t *start,
                                                        CdfMeta *meta) {
    __shared__ T wbuf[CDF_BLK], obuf[CDF_BLK];
    __shared__ Advance wtot[4];
    __shared__ long long base_sh;
    __shared__ int cross_sh, stop_sh;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int64_t first = adv ? (int64_t)meta->first : n;
    int64_t bits = 0;  // the running sum, the same in every thread
    int64_t b = 0;
    while (b < nb && b * CDF_BLK < first) {
        const int e0 = chain_exp<T>(bits);
        if (adv) {
            // as many of the next 64 blocks as stay in this binade
            const int64_t q = b + lane;
            const bool ok = q < nb && bexp[q] == e0;
            Advance a = ok ? adv[q] : Advance{chain_cap<T>(), chain_cap<T>()};
            a = wave_scan_advance<T>(a, lane);
            const int64_t nx = bits + ((bits & 1) ? a.d1 : a.d0);
            const unsigned long long out = __ballot(!ok || (uint64_t)nx >= chain_limit<T>(e0));
            const int f = out ? (int)__builtin_ctzll(out) : 64;
            const int64_t before = (int64_t)__shfl_up((long long)nx, 1);
            if (wave == 0 && lane < f) start[q] = lane == 0 ? bits : before;
            if (f > 0) {
                bits = (int64_t)__shfl((long long)nx, f - 1);
                b += f;
                continue;
            }
        }
        const int64_t i0 = b * CDF_BLK;
        const int64_t left = first - i0;
        int len = left < CDF_BLK ? (int)left : CDF_BLK;
        if (tid == 0) stop_sh = len;
        __syncthreads();  // also: the last block's obuf has been written out
#pragma unroll
        for (int q = 0; q < CDF_PER; ++q) {
            const int i = tid + 256 * q;
            if (i < len) {
                const T x = w[i0 + i];
                if (!(x >= error_if_below)) atomicMin(&stop_sh, i);
                wbuf[i] = x < (T)0 ? (T)0 : x;
            }
        }
        __syncthreads();
        if (stop_sh < len) {
            len = stop_sh;
            first = i0 + len;
        }
        int pos = 0;  // terms of the block already in the sum
        if (b == 0) {
            // the first sums leave a binade every few terms: added one by one
            pos = len < CDF_HEAD ? len : CDF_HEAD;
            if (tid == 0) {
                T s = (T)0;
#pragma unroll 8
                for (int i = 0; i < pos; ++i) {
                    s = s + wbuf[i];
                    obuf[i] = s;
                }
                base_sh = (long long)chain_bits(s);
            }
            __syncthreads();
            bits = (int64_t)base_sh;
            __syncthreads();  // (base_sh is written again below)
        }
        while (true) {
            const int e = chain_exp<T>(bits);
            const uint64_t limit = chain_limit<T>(e);
            Advance t[CDF_PER], a{0, 0};
#pragma unroll
            for (int q = 0; q < CDF_PER; ++q) {
                const int i = CDF_PER * tid + q;
                t[q] = i >= pos && i < len ? chain_term<T>(wbuf[i], e) : Advance{0, 0};
                a = chain_compose<T>(a, t[q]);
            }
            const Advance incl = wave_scan_advance<T>(a, lane);
            Advance excl = shfl_up_advance<T>(incl, 1);
            if (lane == 0) excl = Advance{0, 0};
            if (lane == 63) wtot[wave] = incl;
            if (tid == 0) cross_sh = CDF_BLK;
            __syncthreads();
            Advance pre{0, 0}, tot{0, 0};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (q == wave) pre = tot;
                tot = chain_compose<T>(tot, wtot[q]);
            }
            excl = chain_compose<T>(pre, excl);
            int64_t cur = bits + ((bits & 1) ? excl.d1 : excl.d0);
            int cross = CDF_BLK;
            if ((uint64_t)cur < limit) {
#pragma unroll
                for (int q = 0; q < CDF_PER; ++q) {
                    const int i = CDF_PER * tid + q;
                    if (i >= pos && i < len && cross == CDF_BLK) {
                        const int64_t nx = cur + ((cur & 1) ? t[q].d1 : t[q].d0);
                        if ((uint64_t)nx >= limit) {
                            cross = i;
                        } else {
                            cur = nx;
                            obuf[i] = chain_value<T>(cur);
                        }
                    }
                }
                if (cross < CDF_BLK) atomicMin(&cross_sh, cross);
            }
            __syncthreads();
            const int first_cross = cross_sh;
            if (first_cross == CDF_BLK) {
                bits += (bits & 1) ? tot.d1 : tot.d0;
                break;
            }
            // the term that leaves the binade: one addition in T
            if (cross == first_cross) {
                const T s = chain_value<T>(cur) + wbuf[cross];
                obuf[cross] = s;
                base_sh = (long long)chain_bits(s);
            }
            __syncthreads();
            bits = (int64_t)base_sh;
            pos = first_cross + 1;
        }
        __syncthreads();
        for (int i = tid; i < len; i += 256) w[i0 + i] = obuf[i];
        if (tid == 0) start[b] = -1;
        ++b;
    }
    if (tid == 0) {
        const T sum = chain_value<T>(bits);
        const T floor_sum = (T)sqrt((double)n) * std::numeric_limits<T>::epsilon();
        const bool ok = first == n && sum >= floor_sum;
        meta->first = (long long)first;
        meta->status = first < n ? 1 + (long long)first : (ok ? 0 : -1);
        meta->inv = ok ? (double)((T)1 / sum) : 1.0;
    }
}

// w[i] = partial sum * (1 / sum) (blas::scal), or the plain partial sums
// (inv = 1) when the sums failed
template <typename T>
__global__ __launch_bounds__(256) void cdf_write_kernel(T *w, const int64_t *start, const CdfMeta *meta) {
    __shared__ T buf[CDF_BLK];
    __shared__ Advance wtot[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t i0 = (int64_t)blockIdx.x * CDF_BLK;
    const int64_t left = meta->first - i0;
    if (left <= 0) return;
    const int len = left < CDF_BLK ? (int)left : CDF_BLK;
    const T inv = (T)meta->inv;
    const int64_t bits = start[blockIdx.x];
    if (bits < 0) {
        for (int i = tid; i < len; i += 256) w[i0 + i] = w[i0 + i] * inv;
        return;
    }
    cdf_load_block(w + i0, len, buf, tid);
    __syncthreads();
    const int e = chain_exp<T>(bits);
    Advance t[CDF_PER], a{0, 0};
#pragma unroll
    for (int q = 0; q < CDF_PER; ++q) {
        const int i = CDF_PER * tid + q;
        t[q] = i < len ? chain_term<T>(buf[i], e) : Advance{0, 0};
        a = chain_compose<T>(a, t[q]);
    }
    const Advance incl = wave_scan_advance<T>(a, lane);
    Advance excl = shfl_up_advance<T>(incl, 1);
    if (lane == 0) excl = Advance{0, 0};
    if (lane == 63) wtot[wave] = incl;
    __syncthreads();
    Advance pre{0, 0};
    for (int q = 0; q < wave; ++q) pre = chain_compose<T>(pre, wtot[q]);
    excl = chain_compose<T>(pre, excl);
    int64_t cur = bits + ((bits & 1) ? excl.d1 : excl.d0);
#pragma unroll
    for (int q = 0; q < CDF_PER; ++q) {
        const int i = CDF_PER * tid + q;
        if (i < len) {
            cur += (cur & 1) ? t[q].d1 : t[q].d0;
            buf[i] = chain_value<T>(cur) * inv;
        }
    }
    __syncthreads();
    for (int i = tid; i < len; i += 256) w[i0 + i] = buf[i];
}

static void next_state(const rbx_rng_state *state, uint64_t counters, rbx_rng_state *next) {
    if (next == nullptr) return;
    rbx_rng_state s = *state;
    ctr_to_words(ctr_add(ctr_from_words(s.counter), counters), s.counter);
    *next = s;
}

template <typename T>
static void iid_uniform_impl(int64_t n, int64_t k, int64_t *samples, T *rademachers, const rbx_rng_state *state,
                             rbx_rng_state *next, hipStream_t st) {
    RBX_REQUIRE(state != nullptr);
    RBX_REQUIRE(n >= 0 && k >= 0);
    const int per = rademachers ? 2 : 4;
    const int64_t counters = (k + per - 1) / per;
    if (k > 0) {
        RBX_REQUIRE(samples != nullptr);
        const Ctr128 ctr = ctr_from_words(state->counter);
        const int64_t blocks = (counters + 255) / 256;
        RBX_REQUIRE(blocks < (1ll << 31));
        ProfScope prof("iid_uniform_kernel", st);
        hipLaunchKernelGGL((iid_uniform_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, st, ctr, state->key[0],
                           state->key[1], n, k, samples, rademachers);
        RBX_HIP(hipGetLastError());
    }
    next_state(state, (uint64_t)counters, next);
}

// The draws by a table, where that is faster: arrays of up to 2^16 entries
// (14-62 us against 18-204 us for 10^3 to 2^24 draws from 20000), longer ones
// from a quarter as many draws on (10^6 entries, FP64: 2^17 draws 32 us either
// way, 2^20 36 against 79 us, 2^24 178 against 875 us).  False, with nothing
// launched, for the other sizes and without the memory.
constexpr int64_t CDF_NEAR_MIN = 1 << 16;
template <typename T>
static bool cdf_by_table(int64_t n, const T *cdf, int64_t k, int64_t *samples, Ctr128 ctr, const rbx_rng_state *state,
                         hipStream_t st) {
    if (n < 1 || n >= (int64_t)INT32_MAX || (n > CDF_NEAR_MIN && k < n / 4)) return false;
    const int64_t tb = std::min<int64_t>((std::max<int64_t>(n, CDF_BUCKETS + 1) + 255) / 256, CDF_TABLE_BLOCKS);
    const size_t b_start = (CDF_BUCKETS + 64) * sizeof(uint32_t), b_flags = CDF_TABLE_BLOCKS * sizeof(int);
    const size_t bytes = b_start + b_flags + (size_t)n * sizeof(uint16_t);
    if (!scratch_usable(SCRATCH_SPARSE_G, bytes, st)) return false;
    char *ws;
    try {
        ws = (char *)scratch(SCRATCH_SPARSE_G, bytes, st);
    } catch (const Fail &f) {
        if (f.st != RBX_OUT_OF_MEMORY) throw;
        clear_error();
        return false;
    }
    uint32_t *start = (uint32_t *)ws;
    int *unsorted = (int *)(ws + b_start);
    uint16_t *low = (uint16_t *)(ws + b_start + b_flags);
    hipLaunchKernelGGL((cdf_table_kernel<T>), dim3((unsigned)tb), dim3(256), 0, st, n, cdf, start, low, unsorted);
    const int64_t blocks = std::min<int64_t>((k + 4095) / 4096, num_cus());
    auto draw = [&](auto near) {
        hipLaunchKernelGGL((iid_cdf_table_kernel<T, decltype(near)::value>), dim3((unsigned)blocks), dim3(1024), 0, st,
                           ctr, state->key[0], state->key[1], n, cdf, (const uint32_t *)start, (const uint16_t *)low,
                           (const int *)unsorted, (int)tb, k, samples);
    };
    if (n > CDF_NEAR_MIN) draw(std::true_type{});
    else draw(std::false_type{});
    RBX_HIP(hipGetLastError());
    return true;
}

template <typename T>
static void iid_cdf_impl(int64_t n, const T *cdf, int64_t k, int64_t *samples, const rbx_rng_state *state,
                         rbx_rng_state *next, hipStream_t st) {
    RBX_REQUIRE(state != nullptr);
    RBX_REQUIRE(n >= 0 && k >= 0);
    const int64_t counters = (k + 3) / 4;
    if (k > 0) {
        RBX_REQUIRE(samples != nullptr && (n == 0 || cdf != nullptr));
        const Ctr128 ctr = ctr_from_words(state->counter);
        ProfScope prof("iid_cdf_kernel", st);
        if (cdf_by_table<T>(n, cdf, k, samples, ctr, state, st)) {
            next_state(state, (uint64_t)counters, next);
            return;
        }
        int64_t blocks = (counters + 255) / 256;
        if (blocks > 4 * (int64_t)num_cus()) blocks = 4 * (int64_t)num_cus();
        hipLaunchKernelGGL((iid_cdf_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, st, ctr, state->key[0],
                           state->key[1], n, cdf, k, samples);
        RBX_HIP(hipGetLastError());
    }
    next_state(state, (uint64_t)counters, next);
}

template <typename T>
static void weights_to_cdf_impl(int64_t n, T *w, T error_if_below, hipStream_t st) {
    RBX_REQUIRE(n >= 0);
    RBX_REQUIRE(n == 0 || w != nullptr);
    const int64_t nb = (n + CDF_BLK - 1) / CDF_BLK;
    RBX_REQUIRE(nb < (1ll << 31));
    const bool direct = nb <= CDF_DIRECT;
    // meta | start | adv | prefix | bexp | bbad
    char *ws = (char *)scratch(SCRATCH_SMALL, 64 + (size_t)nb * (8 + 16 + 8 + 4 + 4) + 8, st);
    CdfMeta *meta = (CdfMeta *)ws;
    int64_t *start = (int64_t *)(ws + 64);
    Advance *adv = (Advance *)(start + nb);
    double *bsum = (double *)(adv + nb);
    int *bexp = (int *)(bsum + nb + 1), *bbad = bexp + nb;
    {
        ProfScope prof("weights_to_cdf_kernel", st);
        const dim3 grid((unsigned)nb);
        if (!direct) {
            hipLaunchKernelGGL((cdf_sums_kernel<T>), grid, dim3(256), 0, st, n, (const T *)w, error_if_below, bsum,
                               bbad);
            hipLaunchKernelGGL(cdf_guess_kernel, dim3(1), dim3(1024), 0, st, n, nb, bsum, (const int *)bbad, meta);
            hipLaunchKernelGGL((cdf_advance_kernel<T>), grid, dim3(256), 0, st, (const T *)w, (const double *)bsum,
                               (const CdfMeta *)meta, adv, bexp);
        }
        hipLaunchKernelGGL((cdf_chain_kernel<T>), dim3(1), dim3(256), 0, st, n, w, error_if_below, nb,
                           direct ? (const Advance *)nullptr : (const Advance *)adv, (const int *)bexp, start, meta);
        if (nb > 0)
            hipLaunchKernelGGL((cdf_write_kernel<T>), grid, dim3(256), 0, st, w, (const int64_t *)start,
                               (const CdfMeta *)meta);
        RBX_HIP(hipGetLastError());
    }
    long long h = 0;
    RBX_HIP(hipMemcpyAsync(&h, &meta->status, sizeof(h), hipMemcpyDeviceToHost, st));
    RBX_HIP(hipStreamSynchronize(st));
    if (h > 0)
        RBX_FAIL(RBX_INVALID_ARG, "weights_to_cdf: w[%lld] is below error_if_below = %e", h - 1,
                 (double)error_if_below);
    if (h < 0) RBX_FAIL(RBX_INVALID_ARG, "weights_to_cdf: the weights sum to less than sqrt(n) * epsilon");
}

// ---------------------------------------------------------------- power-law sparse test data
// A random m x n CSR matrix whose column popularity follows a Zipf law (no
// RandBLAS counterpart; RandBLAS's own generators, sparse_data/
// random_matrix.hh:136-358, draw uniform-density matrices from one sequential
// stream).  Built from the library's counter-addressed samplers, so every
// stage is a pure function of (key, counter) and runs in parallel:
//   w[c]  = (c + 1)^(-1 / (exponent - 1))    host libm pow, rounded to T
//   cdf   = weights_to_cdf(w)                 (util.hh:459-472)
//   cols  = sample_indices_iid(n, cdf, k)     from `state`      (util.hh:493-514)
//   rows  = sample_indices_iid_uniform(m, k)  from the state after it (util.hh:516-546)
//   the k (row, column) pairs sorted, repeated pairs kept once -> CSR
//   vals  = the first nnz entries of a DenseDist(nnz, 1) Gaussian operator
//           from the state after the row draws (dense_skops.hh:563-606)
// Row degrees are Binomial(k, 1/m) before merging; the column degrees have a
// power-law tail with the given exponent.

// keys[i] = rows[i] * n + cols[i]
__global__ __launch_bounds__(256) void plc_keys_kernel(const int64_t *rows, const int64_t *cols, int64_t k,
                                                       int64_t n, uint64_t *keys) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < k) keys[i] = (uint64_t)rows[i] * (uint64_t)n + (uint64_t)cols[i];
}

// first[i] = 1 for the first of each run of equal sorted keys
__global__ __launch_bounds__(256) void plc_first_kernel(const uint64_t *keys, int64_t k, int64_t *first) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < k) first[i] = (i == 0 || keys[i] != keys[i - 1]) ? 1 : 0;
}

// Unique entry e = pos[i] (sorted key i opening a run): colidxs[e], and
// rowptr[r] = e for every row r in (row of the previous key, row of key i].
// Rows after the last key's row get nnz (the tail kernel).
__global__ __launch_bounds__(256) void plc_compact_kernel(const uint64_t *keys, const int64_t *first,
                                                          const int64_t *pos, int64_t k, int64_t n,
                                                          int64_t *colidxs, int64_t *rowptr) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= k || first[i] == 0) return;
    const int64_t e = pos[i];
    const uint64_t key = keys[i];
    const int64_t r = (int64_t)(key / (uint64_t)n);
    colidxs[e] = (int64_t)(key - (uint64_t)r * (uint64_t)n);
    const int64_t rp = i == 0 ? -1 : (int64_t)(keys[i - 1] / (uint64_t)n);
    for (int64_t q = rp + 1; q <= r; ++q) rowptr[q] = e;
}

__global__ __launch_bounds__(256) void plc_tail_kernel(const uint64_t *keys, int64_t k, int64_t n, int64_t m,
                                                       const int64_t *first, const int64_t *pos, int64_t *rowptr,
                                                       int64_t *nnz_out) {
    const int64_t r_last = k > 0 ? (int64_t)(keys[k - 1] / (uint64_t)n) : -1;
    const int64_t nnz = k > 0 ? pos[k - 1] + first[k - 1] : 0;
    for (int64_t q = r_last + 1 + (int64_t)threadIdx.x; q <= m; q += blockDim.x) rowptr[q] = nnz;
    if (threadIdx.x == 0) *nnz_out = nnz;
}

static int plc_bits(uint64_t x) {
    int b = 1;
    while (b < 64 && (x >> b) != 0) ++b;
    return b;
}

template <typename T>
static void power_law_csr_impl(int64_t m, int64_t n, int64_t k, double exponent, const rbx_rng_state *state,
                               rbx_csr_matrix *A, rbx_rng_state *next, hipStream_t st) {
    RBX_REQUIRE(state != nullptr && A != nullptr);
    RBX_REQUIRE(m > 0 && n > 0 && k >= 0);
    RBX_REQUIRE(exponent > 1.0);
    RBX_REQUIRE(A->rowptr != nullptr);
    RBX_REQUIRE(k == 0 || (A->colidxs != nullptr && A->vals != nullptr));
    const uint64_t mn = (uint64_t)safe_mul(m, n);
    RBX_REQUIRE(k < (1ll << 31) && mn < (1ull << 63));
    // column weights on the host (libm pow), then the device CDF
    std::vector<T> w((size_t)n);
    const double rank_exp = -1.0 / (exponent - 1.0);
    for (int64_t c = 0; c < n; ++c) w[(size_t)c] = (T)std::pow((double)(c + 1), rank_exp);
    const size_t b_cdf = ((size_t)n * sizeof(T) + 255) / 256 * 256, b_k = ((size_t)(k > 0 ? k : 1) * 8 + 255) / 256 * 256;
    size_t sort_bytes = 0, scan_bytes = 0;
    if (k > 0) {
        RBX_HIP(rocprim::radix_sort_keys(nullptr, sort_bytes, (uint64_t *)nullptr, (uint64_t *)nullptr, (size_t)k, 0,
                                         plc_bits(mn - 1), st));
        RBX_HIP(rocprim::exclusive_scan(nullptr, scan_bytes, (int64_t *)nullptr, (int64_t *)nullptr, (int64_t)0,
                                        (size_t)k, rocprim::plus<int64_t>(), st));
    }
    const size_t b_tmp = ((sort_bytes > scan_bytes ? sort_bytes : scan_bytes) + 255) / 256 * 256;
    char *ws = (char *)scratch(SCRATCH_SPARSE_OP, b_cdf + 5 * b_k + b_tmp + 256, st);
    T *cdf = (T *)ws;
    int64_t *rows = (int64_t *)(ws + b_cdf);
    uint64_t *keys = (uint64_t *)(ws + b_cdf + b_k), *keys2 = (uint64_t *)(ws + b_cdf + 2 * b_k);
    int64_t *first = (int64_t *)(ws + b_cdf + 3 * b_k), *pos = (int64_t *)(ws + b_cdf + 4 * b_k);
    void *tmp = ws + b_cdf + 5 * b_k;
    int64_t *d_nnz = (int64_t *)(ws + b_cdf + 5 * b_k + b_tmp);
    RBX_HIP(hipMemcpyAsync(cdf, w.data(), (size_t)n * sizeof(T), hipMemcpyHostToDevice, st));
    weights_to_cdf_impl<T>(n, cdf, (T)-1, st);  // synchronises the stream (w may go)

    rbx_rng_state s1, s2;
    int64_t *cols = A->colidxs;  // the column draws, overwritten by the merged columns below
    iid_cdf_impl<T>(n, cdf, k, cols, state, &s1, st);
    iid_uniform_impl<T>(m, k, rows, nullptr, &s1, &s2, st);
    const int64_t blocks = (k + 255) / 256;
    if (k > 0) {
        hipLaunchKernelGGL(plc_keys_kernel, dim3((unsigned)blocks), dim3(256), 0, st, rows, cols, k, n, keys);
        RBX_HIP(hipGetLastError());
        RBX_HIP(rocprim::radix_sort_keys(tmp, sort_bytes, keys, keys2, (size_t)k, 0, plc_bits(mn - 1), st));
        hipLaunchKernelGGL(plc_first_kernel, dim3((unsigned)blocks), dim3(256), 0, st, keys2, k, first);
        RBX_HIP(hipGetLastError());
        RBX_HIP(rocprim::exclusive_scan(tmp, scan_bytes, first, pos, (int64_t)0, (size_t)k, rocprim::plus<int64_t>(),
                                        st));
        hipLaunchKernelGGL(plc_compact_kernel, dim3((unsigned)blocks), dim3(256), 0, st, keys2, first, pos, k, n,
                           A->colidxs, A->rowptr);
        RBX_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(plc_tail_kernel, dim3(1), dim3(256), 0, st, keys2, k, n, m, first, pos, A->rowptr, d_nnz);
    RBX_HIP(hipGetLastError());
    int64_t nnz = 0;
    RBX_HIP(hipMemcpyAsync(&nnz, d_nnz, sizeof(nnz), hipMemcpyDeviceToHost, st));
    RBX_HIP(hipStreamSynchronize(st));
    // values: DenseDist(nnz, 1) Gaussian from s2 (natural layout ColMajor:
    // entry i is word i % 4 of counter s2 + i / 4); next = s2 + ceil(nnz / 4)
    rbx_rng_state s3 = s2;
    if (nnz > 0) {
        rbx_dense_skop V{};
        V.dist.n_rows = nnz;
        V.dist.n_cols = 1;
        V.dist.family = 'G';
        V.dist.major_axis = 'L';
        V.seed_state = s2;
        const GenMap g = gen_map(V, 'N', 0, 0, false);
        fill_generated<T>(g, nnz, 1, (T *)A->vals, 1, nnz, st);
        next_state(&s2, (uint64_t)((nnz + 3) / 4), &s3);
    }
    A->n_rows = m;
    A->n_cols = n;
    A->nnz = nnz;
    if (next) *next = s3;
}

}  // namespace rbx

using namespace rbx;

extern "C" {

rbx_status rbx_sample_indices_iid_uniform(int64_t n, int64_t k, int64_t *samples, const rbx_rng_state *state,
                                          rbx_rng_state *next_state_out, void *stream) {
    RBX_API_BEGIN
    iid_uniform_impl<float>(n, k, samples, nullptr, state, next_state_out, (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_ssample_indices_iid_uniform_signed(int64_t n, int64_t k, int64_t *samples, float *rademachers,
                                                  const rbx_rng_state *state, rbx_rng_state *next_state_out,
                                                  void *stream) {
    RBX_API_BEGIN
    RBX_REQUIRE(k == 0 || rademachers != nullptr);
    iid_uniform_impl<float>(n, k, samples, rademachers, state, next_state_out, (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_dsample_indices_iid_uniform_signed(int64_t n, int64_t k, int64_t *samples, double *rademachers,
                                                  const rbx_rng_state *state, rbx_rng_state *next_state_out,
                                                  void *stream) {
    RBX_API_BEGIN
    RBX_REQUIRE(k == 0 || rademachers != nullptr);
    iid_uniform_impl<double>(n, k, samples, rademachers, state, next_state_out, (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_ssample_indices_iid(int64_t n, const float *cdf, int64_t k, int64_t *samples,
                                   const rbx_rng_state *state, rbx_rng_state *next_state_out, void *stream) {
    RBX_API_BEGIN
    iid_cdf_impl<float>(n, cdf, k, samples, state, next_state_out, (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_dsample_indices_iid(int64_t n, const double *cdf, int64_t k, int64_t *samples,
                                   const rbx_rng_state *state, rbx_rng_state *next_state_out, void *stream) {
    RBX_API_BEGIN
    iid_cdf_impl<double>(n, cdf, k, samples, state, next_state_out, (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_spower_law_csr(int64_t m, int64_t n, int64_t k, double exponent, const rbx_rng_state *state,
                              rbx_csr_matrix *A, rbx_rng_state *next_state_out, void *stream) {
    RBX_API_BEGIN
    power_law_csr_impl<float>(m, n, k, exponent, state, A, next_state_out, (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_dpower_law_csr(int64_t m, int64_t n, int64_t k, double exponent, const rbx_rng_state *state,
                              rbx_csr_matrix *A, rbx_rng_state *next_state_out, void *stream) {
    RBX_API_BEGIN
    power_law_csr_impl<double>(m, n, k, exponent, state, A, next_state_out, (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_sweights_to_cdf(int64_t n, float *w, float error_if_below, void *stream) {
    RBX_API_BEGIN
    weights_to_cdf_impl<float>(n, w, error_if_below, (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_dweights_to_cdf(int64_t n, double *w, double error_if_below, void *stream) {
    RBX_API_BEGIN
    weights_to_cdf_impl<double>(n, w, error_if_below, (hipStream_t)stream);
    RBX_API_END
}

}  // extern "C"
