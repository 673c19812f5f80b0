// rbx_bf16.hip -- BF16-split form of the left dense sketch on the gfx950
// BF16 matrix cores (no RandBLAS counterpart; the FP32 analogue is lskge3,
// skge.hh:154-202).
//
//   B = alpha * op(bf16(submat(S))) * op(A) + beta * B
//
// Three kernels:
//   1. split:  op(A) (FP32, any strides) -> T bfloat16 planes A_1..A_T with
//      A = A_1 + ... + A_T + residual.  Every term is the round-to-nearest-even
//      of the previous remainder, and each remainder is exact in FP32.  The
//      planes are stored fragment-packed: for a 32-column block and a 16-deep
//      K step, the 64 lanes' MFMA B operands (8 bf16 each) are one contiguous
//      1 KB run, so every load instruction of the main kernel is a full
//      coalesced 1 KB read.  Zero padding to Kp (multiple of 32) x Np
//      (multiple of 256).
//   2. main:   one 256-thread workgroup per (64-row block, 1024-column block,
//      K-split).  Each 32-wide K-chunk of the operator is generated from its
//      Philox counters, rounded to bfloat16 and double-buffered in LDS; the
//      four waves each own 256 columns and keep a 64 x 256 FP32 accumulator
//      (2 x 8 blocks of v_mfma_f32_32x32x16_bf16, 256 AGPRs).  Each operator
//      entry is generated once per 1024 columns.  B operands rotate through
//      registers: the load of block j for the next K step is issued right
//      after block j's MFMAs of this step, so loads are in flight for a whole
//      step.  The K-split bounds each FP32 accumulation chain; partial tiles
//      go to a row-major scratch.
//   3. reduce: B = alpha * sum_s partial_s (in FP64, fixed order) + beta * B.
// WG-to-tile mapping is XCD-aware: workgroups that share a K-range are
// dispatched to the same XCD back to back, so the A planes they stream are
// served from that XCD's L2.
#include <vector>

#include "rbx_internal.hh"
#include "rbx_gemm_common.hh"
#include "rbx_fastgen.hh"


namespace rbx {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int BF_MT = 64, BF_NT = 1024, BF_KC = 32, BF_LDK = 40, BF_NTHR = 256;


// ---------------------------------------------------------------- split
// Element (k, j) of term t (of T) lives at
//   ((((j/32)*(Kp/16) + k/16)*T + t)*64 + j%32 + 32*((k/8)%2))*8 + k%8,
// i.e. for each 32-column block and 16-deep K step the T terms' 1 KB runs are
// adjacent: a kernel needs one pointer per column block, and the term is a
// constant 1 KB offset.
// One wave per (32-column block cb, 16-deep K step s).  Lane l handles column
// 32*cb + l%32 and k = 16*s + 8*(l/32) .. +7, and writes lane l's 16-byte slot
// of the block's 1 KB run of every term, so the wave's stores are T
// contiguous KB.
__global__ __launch_bounds__(256) void split_kernel(const float *A, int64_t rs, int64_t cs, int64_t K, int64_t N,
                                                    int64_t Kp, int64_t Np, int terms, uint16_t *planes) {
    const int64_t KS = Kp / 16;
    const int64_t n_waves = (Np / 32) * KS;
    const int lane = threadIdx.x & 63;
    const int64_t wave0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t wstride = ((int64_t)gridDim.x * blockDim.x) >> 6;
    for (int64_t w = wave0; w < n_waves; w += wstride) {
        const int64_t cb = w / KS, st = w - cb * KS;
        const int64_t j = cb * 32 + (lane & 31);
        const int64_t k0 = st * 16 + 8 * (lane >> 5);
        uint16_t out[3][8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int64_t k = k0 + e;
            float a = (k < K && j < N) ? A[k * rs + j * cs] : 0.0f;
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                uint16_t h = bf16_rne(a);
                out[t][e] = h;
                a = __fsub_rn(a, bf16_to_f32(h));  // exact
            }
        }
        const int64_t dst = (cb * KS + st) * terms * 512 + lane * 8;
        for (int t = 0; t < terms; ++t) {
            u32x4 v;
            v.x = (uint32_t)out[t][0] | ((uint32_t)out[t][1] << 16);
            v.y = (uint32_t)out[t][2] | ((uint32_t)out[t][3] << 16);
            v.z = (uint32_t)out[t][4] | ((uint32_t)out[t][5] << 16);
            v.w = (uint32_t)out[t][6] | ((uint32_t)out[t][7] << 16);
            *(u32x4 *)(planes + dst + t * 512) = v;
        }
    }
}

// Unit-stride K (column-major A, or row-major A^T): one workgroup per
// (32-column block, 256-deep K range).  Each column's 256 consecutive values
// are one contiguous 1 KB read; the tile is transposed through LDS and then
// written as the block's 16 steps of fragment runs (the layout above).
constexpr int SPL_KT = 256, SPL_LD = 260;
template <bool VEC>
__global__ __launch_bounds__(256) void split_kunit_kernel(const float *A, int64_t cs, int64_t K, int64_t N,
                                                          int64_t Kp, int terms, uint16_t *planes,
                                                          int64_t kt_base) {
    __shared__ __attribute__((aligned(16))) float tile[32][SPL_LD];
    const int tid = threadIdx.x;
    const int64_t KS = Kp / 16;
    const int64_t cb = blockIdx.y;
    const int64_t kt0 = ((int64_t)blockIdx.x + kt_base) * SPL_KT;  // this launch's K tiles start at kt_base
    // load: a wave reads 1 KB runs of one column, k in [kt0, kt0 + 256); all
    // eight of a thread's loads are issued before the first LDS store.
    // VEC: 16-byte loads (A and the column stride are 4-float aligned)
    const int q = tid & 63, c0 = tid >> 6;
    const int64_t k = kt0 + 4 * q;
    float4 v[8];
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        const int64_t j = cb * 32 + c0 + 4 * p;
        const float *src = A + k + j * cs;
        if (VEC && j < N && k + 3 < K) {
            v[p] = *(const float4 *)src;
        } else {
            v[p].x = (j < N && k < K) ? src[0] : 0.0f;
            v[p].y = (j < N && k + 1 < K) ? src[1] : 0.0f;
            v[p].z = (j < N && k + 2 < K) ? src[2] : 0.0f;
            v[p].w = (j < N && k + 3 < K) ? src[3] : 0.0f;
        }
    }
#pragma unroll
    for (int p = 0; p < 8; ++p) *(float4 *)&tile[c0 + 4 * p][4 * q] = v[p];
    __syncthreads();
    // split: lane task (step s, lane l) of this K range, 4 per thread
    const int64_t steps = (KS - kt0 / 16) < 16 ? (KS - kt0 / 16) : 16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int task = tid + 256 * i;
        const int st = task >> 6, l = task & 63;
        if (st >= steps) break;
        const float *src = &tile[l & 31][16 * st + 8 * (l >> 5)];
        // pairs rounded by the hardware RNE conversion (v_cvt_pk_bf16_f32,
        // the same bits as bf16_rne for every non-NaN input), each
        // remainder exact in FP32
        f32x2 a[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) a[p] = f32x2{src[2 * p], src[2 * p + 1]};
        u32x4 out[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector(a[p], bf16x2));
                out[t][p] = h;
                a[p][0] = __fsub_rn(a[p][0], __uint_as_float(h << 16));
                a[p][1] = __fsub_rn(a[p][1], __uint_as_float(h & 0xffff0000u));
            }
        }
        const int64_t dst = (cb * KS + kt0 / 16 + st) * terms * 512 + l * 8;
        for (int t = 0; t < terms; ++t) *(u32x4 *)(planes + dst + t * 512) = out[t];
    }
}

struct Bf16Problem {
    int64_t M, N, K, Kp, Np;
    GenMap g;
    const uint16_t *planes;  // fragment-packed terms (see split_kernel)
    float *part;  // nS x M x ldp, row-major
    int64_t ldp;  // N rounded up to a multiple of 4
    int64_t kw;   // K per split (multiple of BF_KC)
    int nMB, nNB, nS;  // row blocks, column blocks and K-splits of the launch
    int sp0;      // first K-split of the launch
};

// 32x32 output block, element r of lane l: row 8*(r/4) + 4*(l/32) + r%4, column l%32.
__device__ __forceinline__ int out_row32(int lane, int r) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// The form for operators whose counters run along the output rows or whose
// window starts inside a counter; every other call takes the pair kernel.
template <int TERMS>
__global__ __launch_bounds__(BF_NTHR, 1) void bf16_skge_kernel(Bf16Problem pb) {
    __shared__ __attribute__((aligned(16))) uint16_t Ss[2][BF_MT * BF_LDK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    // XCD-aware tile order: consecutive tiles (same K-split) land on one XCD
    const int W = pb.nMB * pb.nNB * pb.nS;
    const int L = blockIdx.x;
    const int t = (W % 8 == 0) ? (L % 8) * (W / 8) + L / 8 : L;
    const int mb = t % pb.nMB;
    const int rest = t / pb.nMB;
    const int nb = rest % pb.nNB;
    const int sp = rest / pb.nNB;
    const int64_t m0 = (int64_t)mb * BF_MT;
    const int64_t n0 = (int64_t)nb * BF_NT;
    const int64_t kbeg = (int64_t)sp * pb.kw;
    int64_t kend = kbeg + pb.kw;
    if (kend > pb.Kp) kend = pb.Kp;
    const int nchunks = (int)((kend - kbeg) / BF_KC);
    const GenMap g = pb.g;

    f32x16 acc[2][8];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    const int64_t wcol = n0 + wave * 256;        // first column of this wave
    const bool active = wcol < pb.Np;    // Np is a multiple of 256: all 8 blocks or none
    const int64_t KS = pb.Kp / 16;
    // lane's B operand for block j, K step s, term t:
    //   planes + (((wcol/32 + j)*KS + s)*TERMS + t)*512 + lane*8
    const uint16_t *bbase = pb.planes + (wcol >> 5) * KS * (TERMS * 512) + lane * 8;
    const int64_t bstep_blk = KS * (TERMS * 512);  // elements between column blocks
    const int64_t s_first = kbeg / 16, s_last = kend / 16 - 1;

    auto gen_chunk = [&](int c, uint16_t *lds) {
        gen_tile<uint16_t, BF_MT, BF_KC, BF_NTHR>(g, m0, kbeg + (int64_t)c * BF_KC, pb.M, pb.K, lds, BF_LDK, 1, tid);
    };

    bf16x8 bq[8][TERMS];
    if (active) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int tt = 0; tt < TERMS; ++tt)
                bq[j][tt] = __builtin_bit_cast(
                    bf16x8, *(const u32x4 *)(bbase + j * bstep_blk + s_first * (TERMS * 512) + tt * 512));
    }

    if (nchunks > 0) gen_chunk(0, Ss[0]);
    __syncthreads();

    for (int c = 0; c < nchunks; ++c) {
        const int64_t kc = kbeg + (int64_t)c * BF_KC;
        if (c + 1 < nchunks) gen_chunk(c + 1, Ss[(c + 1) & 1]);
        const uint16_t *S = Ss[c & 1];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int koff = ks * 16 + 8 * (lane >> 5);
            const bf16x8 a0 = __builtin_bit_cast(bf16x8, *(const u32x4 *)(S + (lane & 31) * BF_LDK + koff));
            const bf16x8 a1 = __builtin_bit_cast(bf16x8, *(const u32x4 *)(S + (32 + (lane & 31)) * BF_LDK + koff));
            int64_t s_next = kc / 16 + ks + 1;
            if (s_next > s_last) s_next = s_last;  // redundant in-range reload at the end
            if (active) {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
#pragma unroll
                    for (int tt = 0; tt < TERMS; ++tt) {
                        acc[0][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, bq[j][tt], acc[0][j], 0, 0, 0);
                        acc[1][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, bq[j][tt], acc[1][j], 0, 0, 0);
                    }
#pragma unroll
                    for (int tt = 0; tt < TERMS; ++tt)
                        bq[j][tt] = __builtin_bit_cast(
                            bf16x8, *(const u32x4 *)(bbase + j * bstep_blk + s_next * (TERMS * 512) + tt * 512));
                    // keep the reload of block j here, a whole step ahead of
                    // its use: without the barrier the scheduler sinks it
                    // next to the use and every block waits out the latency
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        __syncthreads();
    }

    // partial tile -> scratch (row-major M x N per split; lanes walk columns)
    if (!active) return;
    float *P = pb.part + (int64_t)sp * pb.M * pb.ldp;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t gi = m0 + i * 32 + out_row32(lane, r);
                const int64_t gj = wcol + j * 32 + (lane & 31);
                if (gi < pb.M && gj < pb.ldp) P[gi * pb.ldp + gj] = acc[i][j][r];
            }
}

// Two waves per SIMD.  A 512-thread workgroup owns a
// (32 RB) x (256 CB) output tile; each of its 8 waves owns all 32 RB rows and
// 32 CB columns of it (RB x CB blocks of 32 x 32, 16 RB CB accumulator
// registers, so two waves fit on a SIMD).  The B operands a wave streams per
// 16-deep step are CB x TERMS runs of 1 KB, so the global-load volume per
// MFMA falls as RB grows; the operator rows are generated once per
// workgroup, so generation per output column grows as CB shrinks.  Every
// thread generates RB/2 Philox cells of the next 32-deep chunk per chunk;
// waves 0-3 generate before their MFMAs and waves 4-7 after them, so the two
// waves sharing a SIMD (w and w + 4) are in opposite phases.  Any sizes: the
// planes hold zeros past K and N (the operator entries there are whatever the
// counters give), rows past M are not stored.  The operator's rows run along K
// from a counter boundary.
constexpr int BF_FTHR = 512;
#ifndef RBX_BF16_TALL_RB
#define RBX_BF16_TALL_RB 2
#endif
constexpr int BF_RB = RBX_BF16_TALL_RB, BF_CB = 8 / BF_RB;  // blocks per wave: RB x CB = 8
static_assert(32 * BF_RB == BF_MT, "both kernels' row blocks are the same");
// Wave priority while a wave issues its MFMAs (0: unchanged).
#ifndef RBX_BF16_PRIO
#define RBX_BF16_PRIO 1
#endif

// B-operand buffering depth of the pair kernel, in 16-deep K steps.
#ifndef RBX_BF16_BD
#define RBX_BF16_BD 1
#endif
// K depth of the operator chunks the pair kernel generates per barrier.
#ifndef RBX_BF16_KC
#define RBX_BF16_KC 32
#endif
constexpr int PKC = RBX_BF16_KC, PLDK = PKC + 8, PCPR = PKC / 4;  // PCPR: Philox cells per operator row

template <int TERMS, bool GAUSS, int RB, int CB>
__global__ __launch_bounds__(BF_FTHR, 1) void bf16_skge_pair_kernel(Bf16Problem pb) {
    constexpr int MT = 32 * RB, NT = 256 * CB;
    constexpr int RPP = BF_FTHR / PCPR, NCELL = MT / RPP;  // rows per generation pass, cells per thread
    __shared__ __attribute__((aligned(16))) uint16_t Ss[2][MT * PLDK];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // XCD-aware tile order: consecutive tiles (same K-split) land on one XCD
    const int W = pb.nMB * pb.nNB * pb.nS;
    const int L = blockIdx.x;
    const int t = (W % 8 == 0) ? (L % 8) * (W / 8) + L / 8 : L;
    const int mb = t % pb.nMB;
    const int rest = t / pb.nMB;
    const int nb = rest % pb.nNB;
    const int sp = rest / pb.nNB + pb.sp0;
    const int64_t m0 = (int64_t)mb * MT;
    const int64_t n0 = (int64_t)nb * NT;
    const int64_t kbeg = (int64_t)sp * pb.kw;
    int64_t kend = kbeg + pb.kw;
    if (kend > pb.Kp) kend = pb.Kp;
    const int nchunks = (int)((kend - kbeg) / PKC);
    const GenMap g = pb.g;

    f32x16 acc[RB][CB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    const int64_t wcol = n0 + wave * (32 * CB);
    const int64_t KS = pb.Kp / 16;
    const int64_t bstep_blk = KS * (TERMS * 512);
    // lane's B operand for block j, K step s, term t:
    //   planes + (((wcol/32 + j)*KS + s)*TERMS + t)*512 + lane*8
    const uint16_t *bbase = pb.planes + (wcol >> 5) * KS * (TERMS * 512);
    const uint32_t boff = lane * 16;  // bytes
    // B operand of a block's step (its terms' runs start at the scalar `run`):
    // the lane's offset is the load's own 32-bit one, no vector address arithmetic
    typedef const __attribute__((address_space(1))) char *gptr;
    auto load_b = [&](gptr run, int tt) {
        typedef const __attribute__((address_space(1))) u32x4 *gvec;
        return __builtin_bit_cast(bf16x8, *(gvec)(run + boff + tt * 1024));
    };
    auto run_of = [&](int j, int64_t s) {
        gptr run = (gptr)(bbase + j * bstep_blk + s * (TERMS * 512));
        asm("" : "+s"(run));  // keeps the scalar and the lane's part apart
        return run;
    };
    const int64_t s_first = kbeg / 16, s_last = kend / 16 - 1;

    // generator: thread owns cell (tid % PCPR) of operator rows tid / PCPR + RPP i
    const int frow = tid / PCPR, fcell = tid % PCPR;
    const uint64_t foff = (uint64_t)((g.a_off + m0 + frow) * g.P + ((g.b_off + kbeg) >> 2) + fcell);
    auto gen_chunk = [&](int c, uint16_t *lds) {
#pragma unroll
        for (int i = 0; i < NCELL; ++i) {
            *(uint2 *)(lds + (frow + RPP * i) * PLDK + fcell * 4) = gen4_bf16<GAUSS>(
                ctr_add(g.ctr, foff + (uint64_t)(RPP * i) * g.P + (uint64_t)PCPR * (uint64_t)c), g.k0, g.k1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // first B operands, loaded term-major: the order the loop reloads them
    // in, so the wait before each MFMA group covers only that group's load
    // B operands, BD steps deep: step s uses buffer s % BD (BD divides the
    // chunk's two steps), reloaded right after its MFMAs with step s + BD
    constexpr int BD = RBX_BF16_BD;
    static_assert(BD == 1 || BD == 2, "B operand depth");
    bf16x8 bq[BD][CB][TERMS];
#pragma unroll
    for (int bd = 0; bd < BD; ++bd)
#pragma unroll
        for (int tt = 0; tt < TERMS; ++tt)
#pragma unroll
            for (int j = 0; j < CB; ++j) {
                int64_t s_ld = s_first + bd;
                if (s_ld > s_last) s_ld = s_last;
                bq[bd][j][tt] = load_b(run_of(j, s_ld), tt);
                __builtin_amdgcn_sched_barrier(0);
            }

    // one 16-deep K step: block j's B operands for step s + BD are reloaded
    // right after its MFMAs, BD steps ahead of their use
    auto load_a = [&](const uint16_t *S, int ks, bf16x8 *a) {
        const int koff = ks * 16 + 8 * (lane >> 5);
#pragma unroll
        for (int i = 0; i < RB; ++i)
            a[i] = __builtin_bit_cast(bf16x8, *(const u32x4 *)(S + (32 * i + (lane & 31)) * PLDK + koff));
    };
    auto step = [&](const bf16x8 *a, int ks, int64_t s_next) {
        const int bb = ks % BD;
#if RBX_BF16_PRIO
        __builtin_amdgcn_s_setprio(RBX_BF16_PRIO);
#endif
        gptr run[CB];
#pragma unroll
        for (int j = 0; j < CB; ++j) run[j] = run_of(j, s_next);
        // term-outer: consecutive MFMAs on one accumulator are RB x CB apart,
        // and each accumulator still adds its terms in order hi, lo, lo2
#pragma unroll
        for (int tt = 0; tt < TERMS; ++tt) {
#pragma unroll
            for (int j = 0; j < CB; ++j) {
#pragma unroll
                for (int i = 0; i < RB; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], bq[bb][j][tt], acc[i][j], 0, 0, 0);
                // after the MFMAs, into the registers they read: moved ahead of
                // them it would take others (256 and spills)
                __builtin_amdgcn_sched_barrier(0);
                bq[bb][j][tt] = load_b(run[j], tt);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#if RBX_BF16_PRIO
        __builtin_amdgcn_s_setprio(0);
#endif
    };

    const bool late = (wave & 4) != 0;
    gen_chunk(0, Ss[0]);
    __syncthreads();
    for (int c = 0; c < nchunks; ++c) {
        const uint16_t *S = Ss[c & 1];
        uint16_t *Sn = Ss[(c + 1) & 1];
        const int64_t s0 = s_first + (PKC / 16) * c;
        const bool more = c + 1 < nchunks;
        if (more && !late) gen_chunk(c + 1, Sn);
        // both steps' operator fragments are read from LDS up front, so the
        // second step's reads overlap the first step's MFMAs
        bf16x8 a[PKC / 16][RB];
#pragma unroll
        for (int ks = 0; ks < PKC / 16; ++ks) load_a(S, ks, a[ks]);
#pragma unroll
        for (int ks = 0; ks < PKC / 16; ++ks) step(a[ks], ks, s0 + ks + BD > s_last ? s_last : s0 + ks + BD);
        if (more && late) gen_chunk(c + 1, Sn);
        __syncthreads();
    }

    // partial tile -> scratch (row-major M x N per split; lanes walk columns)
    float *P = pb.part + (int64_t)sp * pb.M * pb.ldp;
    const bool inner = m0 + MT <= pb.M && n0 + NT <= pb.ldp;
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t gi = m0 + i * 32 + out_row32(lane, r);
                const int64_t gj = wcol + j * 32 + (lane & 31);
                if (inner || (gi < pb.M && gj < pb.ldp)) P[gi * pb.ldp + gj] = acc[i][j][r];
            }
}

// B[i,j] = alpha * sum_s part[s][i*ldp + j] + beta * B[i*brs + j*bcs], sums in
// FP64 in split order.  RED_R x RED_C tiles (8 x 128): each row of a tile is
// one 512-byte run of every partial (FP32), long enough for full HBM bursts;
// a column-major B is written along i after a transpose through LDS.  A 1-D
// grid of tiles, row-tile major.  With pre != nullptr the sums start from
// pre[i*ldp + j], the FP64 sum of splits 0 .. s0 - 1 (bf16_presum_kernel), and
// continue with split s0: the same additions in the same order.
constexpr int RED_R = 8, RED_C = 128;
__global__ __launch_bounds__(256) void bf16_reduce_kernel(const float *part, int nS, int64_t M, int64_t N, int64_t ldp,
                                                          double alpha, double beta, float *B, int64_t brs,
                                                          int64_t bcs, const double *pre, int s0) {
    __shared__ double tile[RED_R][RED_C + 1];
    const int64_t ntc = (N + RED_C - 1) / RED_C;
    const int64_t i0 = (int64_t)(blockIdx.x / ntc) * RED_R, j0 = (int64_t)(blockIdx.x % ntc) * RED_C;
    const int64_t total = M * ldp;
    {
        // thread: row r, columns c4 .. c4 + 3, 16-byte loads; eight splits'
        // loads are issued together and every sum stays in split order
        typedef float pt4 __attribute__((ext_vector_type(4)));
        const int r = threadIdx.x / (RED_C / 4), c4 = 4 * (threadIdx.x % (RED_C / 4));
        const int64_t i = i0 + r, j = j0 + c4;
        double v[4] = {0.0, 0.0, 0.0, 0.0};
        if (i < M && j < ldp) {
            if (pre != nullptr)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = pre[i * ldp + j + e];
            const float *p = part + i * ldp + j;
            int s = s0;
            for (; s + 8 <= nS; s += 8) {
                pt4 x[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) x[u] = *(const pt4 *)(p + (int64_t)(s + u) * total);
#pragma unroll
                for (int u = 0; u < 8; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] += (double)x[u][e];
            }
            for (; s < nS; ++s) {
                const pt4 x = *(const pt4 *)(p + (int64_t)s * total);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += (double)x[e];
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) tile[r][c4 + e] = v[e];
    }
    __syncthreads();
    const bool cm = brs == 1;
#pragma unroll
    for (int q = 0; q < RED_R * RED_C / 256; ++q) {
        // column-major: consecutive threads walk i; row-major: they walk j
        const int e = threadIdx.x + 256 * q;
        const int ti = cm ? e % RED_R : e / RED_C, tj = cm ? e / RED_R : e % RED_C;
        const int64_t i = i0 + ti, j = j0 + tj;
        if (i < M && j < N) {
            const double v = tile[ti][tj];
            float *b = B + i * brs + j * bcs;
            double out = alpha * v;
            if (beta != 0.0) out += beta * (double)(*b);
            *b = (float)out;
        }
    }
}

// pre[e] = sum of part[s][e] over s = 0 .. ns - 1 in split order, FP64: the
// first splits of bf16_reduce_kernel's sums, run on a helper stream while the
// last K range is still being multiplied.  Lean (four elements and four
// partial loads in flight per thread), so its waves fit in the registers the
// main kernel leaves free on each SIMD.
typedef float pf32x4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void bf16_presum_kernel(const float *part, int ns, int64_t MN, double *pre) {
    const int64_t n4 = MN / 4;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n4; q += (int64_t)gridDim.x * blockDim.x) {
        const pf32x4 *p = (const pf32x4 *)part + q;
        double v0 = 0.0, v1 = 0.0, v2 = 0.0, v3 = 0.0;
        int s = 0;
        for (; s + 4 <= ns; s += 4) {
            pf32x4 x[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] = __builtin_nontemporal_load(p + (int64_t)(s + u) * n4);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                v0 += (double)x[u][0];
                v1 += (double)x[u][1];
                v2 += (double)x[u][2];
                v3 += (double)x[u][3];
            }
        }
        for (; s < ns; ++s) {
            const pf32x4 x = __builtin_nontemporal_load(p + (int64_t)s * n4);
            v0 += (double)x[0];
            v1 += (double)x[1];
            v2 += (double)x[2];
            v3 += (double)x[3];
        }
        double *o = pre + 4 * q;
        o[0] = v0;
        o[1] = v1;
        o[2] = v2;
        o[3] = v3;
    }
}

// 1-D grid of bf16_reduce_kernel over an M x N output
static dim3 reduce_grid(int64_t M, int64_t N) {
    const int64_t nt = ((M + RED_R - 1) / RED_R) * ((N + RED_C - 1) / RED_C);
    RBX_REQUIRE(nt < (1ll << 31));
    return dim3((unsigned)nt);
}

template <int CB>
static void launch_pair(int n_terms, bool gs, dim3 grid, const Bf16Problem &q, hipStream_t stream) {
    if (n_terms == 1 && gs) hipLaunchKernelGGL((bf16_skge_pair_kernel<1, true, BF_RB, CB>), grid, dim3(BF_FTHR), 0, stream, q);
    else if (n_terms == 1) hipLaunchKernelGGL((bf16_skge_pair_kernel<1, false, BF_RB, CB>), grid, dim3(BF_FTHR), 0, stream, q);
    else if (n_terms == 2 && gs) hipLaunchKernelGGL((bf16_skge_pair_kernel<2, true, BF_RB, CB>), grid, dim3(BF_FTHR), 0, stream, q);
    else if (n_terms == 2) hipLaunchKernelGGL((bf16_skge_pair_kernel<2, false, BF_RB, CB>), grid, dim3(BF_FTHR), 0, stream, q);
    else if (gs) hipLaunchKernelGGL((bf16_skge_pair_kernel<3, true, BF_RB, CB>), grid, dim3(BF_FTHR), 0, stream, q);
    else hipLaunchKernelGGL((bf16_skge_pair_kernel<3, false, BF_RB, CB>), grid, dim3(BF_FTHR), 0, stream, q);
    RBX_HIP(hipGetLastError());
}

static void bf16_split_sketch(char layout, char opS, char opA, int64_t d, int64_t n, int64_t m, float alpha,
                              const rbx_dense_skop *S, int64_t ro_s, int64_t co_s, const float *A, int64_t lda,
                              float beta, float *B, int64_t ldb, int n_terms, hipStream_t stream) {
    RBX_REQUIRE(S != nullptr);
    check_layout(layout);
    check_op(opS);
    check_op(opA);
    RBX_REQUIRE(n_terms >= 1 && n_terms <= 3);
    RBX_REQUIRE(d >= 0 && n >= 0 && m >= 0);
    RBX_REQUIRE(ro_s >= 0 && co_s >= 0);
    if (S->buff != nullptr)
        RBX_FAIL(RBX_UNSUPPORTED, "bf16split: only generated operators (S.buff == NULL) are supported");
    DenseGeom geo = dense_geom(S->dist);
    safe_mul(geo.dim_minor, geo.P);
    int64_t rows_S = opS == 'N' ? d : m, cols_S = opS == 'N' ? m : d;
    RBX_REQUIRE(S->dist.n_rows >= rows_S + ro_s);
    RBX_REQUIRE(S->dist.n_cols >= cols_S + co_s);
    int64_t rows_A = opA == 'N' ? m : n, cols_A = opA == 'N' ? n : m;
    if (layout == 'C') {
        RBX_REQUIRE(lda >= rows_A);
        RBX_REQUIRE(ldb >= d);
    } else {
        RBX_REQUIRE(lda >= cols_A);
        RBX_REQUIRE(ldb >= n);
    }
    const int64_t M = d, N = n, K = m;
    const int64_t brs = layout == 'C' ? 1 : ldb, bcs = layout == 'C' ? ldb : 1;
    if (M == 0 || N == 0) return;
    if (alpha == 0.0f || K == 0) {
        scale_output<float>(B, M, N, brs, bcs, beta, stream);
        return;
    }
    // op(A)[k, j] strides
    int64_t ars, acs;
    if (layout == 'C') {
        ars = opA == 'N' ? 1 : lda;
        acs = opA == 'N' ? lda : 1;
    } else {
        ars = opA == 'N' ? lda : 1;
        acs = opA == 'N' ? 1 : lda;
    }
    Bf16Problem pb{};
    pb.M = M;
    pb.N = N;
    pb.K = K;
    pb.Kp = (K + BF_KC - 1) / BF_KC * BF_KC;
    pb.g = gen_map(*S, opS, ro_s, co_s, false);
    // The pair kernel's tile is 256 cb columns wide.  A 32-deep chunk of a tile
    // costs its MFMAs (also for the zero columns past N) and the operator's
    // generation, about as much as those of 160 columns with three terms; the
    // split of a column costs about 4.5 row tiles' MFMAs on it (1.8 ps an entry
    // against 0.4: few output rows with many zero columns pay for it, 147 x
    // 111947 times 616 columns: 488 us in one tile of 1024, 378 in three of 256).
    const bool pair = !pb.g.b_along_rows && (pb.g.b_off & 3) == 0;
    const int64_t row_tiles = (M + BF_MT - 1) / BF_MT;
    int cb = BF_NT / 256;
    if (pair) {
        int64_t best = 0;
        for (int c = BF_CB; c >= 1; c /= 2) {
            const int64_t nb = (N + 256 * c - 1) / (256 * c);
            const int64_t cost = row_tiles * nb * (256 * c * n_terms + 480) + 14 * 256 * c * nb;
            if (c > 1 && nb * 8 * c > 65535) continue;  // the split's grid
            if (best == 0 || cost < best) {
                best = cost;
                cb = c;
            }
        }
    }
    pb.nMB = (int)row_tiles;
    pb.nNB = (int)((N + 256 * cb - 1) / (256 * cb));
    pb.Np = pair ? (int64_t)pb.nNB * 256 * cb : (N + 255) / 256 * 256;
    pb.ldp = (N + 3) / 4 * 4;
    // K per split: bounded FP32 accumulation chains, and enough workgroups
    int64_t kw = 4096;
    int64_t tiles = (int64_t)pb.nMB * pb.nNB;
    int64_t want_splits = (4 * (int64_t)num_cus() + tiles - 1) / tiles;
    int64_t kw_fill = (pb.Kp + want_splits - 1) / want_splits;
    if (kw_fill < kw) kw = kw_fill;
    kw = (kw + PKC - 1) / PKC * PKC;  // a whole number of the pair kernel's chunks (and of BF_KC)
    if (kw < PKC) kw = PKC;
    pb.kw = kw;
    pb.nS = (int)((pb.Kp + kw - 1) / kw);
    RBX_REQUIRE((int64_t)pb.nMB * pb.nNB * pb.nS < (1ll << 31));


    const bool vec = acs % 4 == 0 && ((uintptr_t)A & 15) == 0;
    const int64_t kt_total = (pb.Kp + SPL_KT - 1) / SPL_KT;
    RBX_REQUIRE(kt_total < (1ll << 31) && pb.Np / 32 <= 65535);
    // unit-stride K: coalesced column reads, transposed through LDS; K tiles
    // [kt_first, kt_first + kt_count) on stream s
    auto split_kunit = [&](int64_t kt_first, int64_t kt_count, hipStream_t s) {
        ProfScope prof("bf16_split_kernel", s);
        const dim3 grid((unsigned)kt_count, (unsigned)(pb.Np / 32));
        if (vec)
            hipLaunchKernelGGL(split_kunit_kernel<true>, grid, dim3(256), 0, s, A, acs, K, N, pb.Kp, n_terms,
                               (uint16_t *)pb.planes, kt_first);
        else
            hipLaunchKernelGGL(split_kunit_kernel<false>, grid, dim3(256), 0, s, A, acs, K, N, pb.Kp, n_terms,
                               (uint16_t *)pb.planes, kt_first);
        RBX_HIP(hipGetLastError());
    };
    // the two-wave kernel over K-splits [sp_first, sp_first + sp_count)
    auto main_fast = [&](int sp_first, int sp_count) {
        ProfScope prof("bf16_skge_kernel", stream);
        Bf16Problem q = pb;
        q.sp0 = sp_first;
        q.nS = sp_count;
        const dim3 grid((unsigned)(q.nMB * q.nNB * q.nS));
        const bool gs = q.g.gauss != 0;
        if (cb == BF_CB) launch_pair<BF_CB>(n_terms, gs, grid, q, stream);
        else if (cb == BF_CB / 2) launch_pair<(BF_CB / 2 > 0 ? BF_CB / 2 : 1)>(n_terms, gs, grid, q, stream);
        else launch_pair<(BF_CB / 4 > 0 ? BF_CB / 4 : 1)>(n_terms, gs, grid, q, stream);
    };
    // K-range pipeline of the pair kernel: the split of later K ranges runs on the workspace's helper stream while the
    // main kernel multiplies earlier ones (the split's lean waves fit beside
    // the main kernel's on each CU); the caller's stream waits for each range's
    // split before that range's product, so all helper work is joined before
    // the reduction.
    const int64_t tiles_per_split = pb.kw / SPL_KT;
    const bool pipelined = ars == 1 && pair && pb.nS >= 8 && pb.kw % SPL_KT == 0;
    // the pipeline also sums the first K ranges' partials on the helper
    // stream during the last range's product (FP64, M x N)
    const size_t plane_elems = (size_t)safe_mul(pb.Kp, pb.Np);
    const size_t planes_bytes = ((size_t)n_terms * plane_elems * 2 + 255) / 256 * 256;
    const size_t part_bytes = ((size_t)safe_mul(safe_mul(pb.nS, M), pb.ldp) * 4 + 255) / 256 * 256;
    const size_t pre_bytes = pipelined ? (size_t)safe_mul(M, pb.ldp) * 8 : 0;
    char *ws = (char *)scratch(SCRATCH_BF16, planes_bytes + part_bytes + pre_bytes, stream);
    pb.planes = (const uint16_t *)ws;
    pb.part = (float *)(ws + planes_bytes);
    double *pre = pipelined ? (double *)(ws + planes_bytes + part_bytes) : nullptr;
    int pre_splits = 0;  // splits already in pre
    if (pipelined) {
        // four equal K ranges: only the first range's split runs alone (at the
        // headline shape 7.34 ms per step against 7.62 without the pipeline;
        // an eighth then seven eighths measured 7.38 ms)
        constexpr int NCH = 4;
        int sb[NCH + 1];
        for (int c = 0; c <= NCH; ++c) sb[c] = (int)((int64_t)pb.nS * c / NCH);
        auto kt_of = [&](int sp) { return (int64_t)sp * tiles_per_split < kt_total ? (int64_t)sp * tiles_per_split
                                                                                   : kt_total; };
        hipStream_t hs = ws_aux_stream(stream);
        split_kunit(kt_of(sb[0]), kt_of(sb[1]) - kt_of(sb[0]), stream);
        hipEvent_t fork = ws_event(stream, 0);
        RBX_HIP(hipEventRecord(fork, stream));
        RBX_HIP(hipStreamWaitEvent(hs, fork, 0));
        for (int c = 1; c < NCH; ++c) {
            split_kunit(kt_of(sb[c]), kt_of(sb[c + 1]) - kt_of(sb[c]), hs);
            RBX_HIP(hipEventRecord(ws_event(stream, c), hs));
        }
        for (int c = 0; c < NCH; ++c) {
            if (c > 0) RBX_HIP(hipStreamWaitEvent(stream, ws_event(stream, c), 0));
            main_fast(sb[c], sb[c + 1] - sb[c]);
            if (c == NCH - 2) {
                // partials of ranges 0 .. NCH - 2 are complete: sum them on
                // the helper stream while the last range is multiplied
                hipEvent_t ready = ws_event(stream, NCH);
                RBX_HIP(hipEventRecord(ready, stream));
                RBX_HIP(hipStreamWaitEvent(hs, ready, 0));
                pre_splits = sb[NCH - 1];
                ProfScope prof("bf16_presum_kernel", hs);
                hipLaunchKernelGGL(bf16_presum_kernel, dim3((unsigned)num_cus() * 4), dim3(256), 0, hs,
                                   (const float *)pb.part, pre_splits, M * pb.ldp, pre);
                RBX_HIP(hipGetLastError());
                RBX_HIP(hipEventRecord(ws_event(stream, NCH + 1), hs));
            }
        }
        RBX_HIP(hipStreamWaitEvent(stream, ws_event(stream, NCH + 1), 0));
    } else {
        if (ars == 1) {
            split_kunit(0, kt_total, stream);
        } else {
            int64_t total = (pb.Np / 32) * (pb.Kp / 16) * 64;  // one wave per (block, K step)
            int64_t blocks = (total + 255) / 256;
            if (blocks > 65536) blocks = 65536;
            ProfScope prof("bf16_split_kernel", stream);
            hipLaunchKernelGGL(split_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, A, ars, acs, K, N, pb.Kp,
                               pb.Np, n_terms, (uint16_t *)pb.planes);
            RBX_HIP(hipGetLastError());
        }
        if (pair) {
            main_fast(0, pb.nS);
        } else {
            ProfScope prof("bf16_skge_kernel", stream);
            const dim3 grid((unsigned)(pb.nMB * pb.nNB * pb.nS));
            if (n_terms == 1) hipLaunchKernelGGL((bf16_skge_kernel<1>), grid, dim3(BF_NTHR), 0, stream, pb);
            else if (n_terms == 2) hipLaunchKernelGGL((bf16_skge_kernel<2>), grid, dim3(BF_NTHR), 0, stream, pb);
            else hipLaunchKernelGGL((bf16_skge_kernel<3>), grid, dim3(BF_NTHR), 0, stream, pb);
            RBX_HIP(hipGetLastError());
        }
    }
    {
        const dim3 grid = reduce_grid(M, N);
        ProfScope prof("bf16_reduce_kernel", stream);
        hipLaunchKernelGGL(bf16_reduce_kernel, grid, dim3(256), 0, stream, (const float *)pb.part, pb.nS, M, N, pb.ldp,
                           (double)alpha, (double)beta, B, brs, bcs, (const double *)pre, pre_splits);
        RBX_HIP(hipGetLastError());
    }
}

// ---------------------------------------------------------------- fast generator bounds
// Measures, over every 32-bit word, the distance of the hardware factors of
// the fast generator from the portable factors that define the operator:
//   out[4 b + 0] = max |s' - s|,  out[4 b + 1] = max |c' - c|   (w as w0)
//   out[4 b + 2] = max |r' - r| / r over r > 0                    (w as w1)
//   out[4 b + 3] = number of words with (r' == 0) != (r == 0)
// per workgroup b; the host takes the maxima.  Word w = i + stride * j for
// thread i of the grid, so every word is visited exactly once.
constexpr int FGB_BLOCKS = 16384, FGB_THREADS = 256;
__global__ __launch_bounds__(FGB_THREADS) void fastgen_bounds_kernel(double *out) {
    __shared__ double red[4][FGB_THREADS];
    const uint32_t stride = (uint32_t)FGB_BLOCKS * FGB_THREADS;  // 2^22
    const uint32_t i = blockIdx.x * FGB_THREADS + threadIdx.x;
    double es = 0.0, ec = 0.0, er = 0.0;
    double zero_mismatch = 0.0;
    for (uint32_t j = 0; j < (1u << 10); ++j) {  // 2^22 * 2^10 = 2^32 words
        const uint32_t w = i + stride * j;
        float sf, cf;
        fast_sincos_factor(w, sf, cf);
        float s, c;
        bm_sincos(w, s, c);
        es = fmax(es, fabs((double)sf - (double)s));
        ec = fmax(ec, fabs((double)cf - (double)c));
        const float rf = fast_radius_factor(w);
        const float r = bm_radius(w);
        if (r > 0.0f) er = fmax(er, fabs((double)rf - (double)r) / (double)r);
        if ((rf == 0.0f) != (r == 0.0f)) zero_mismatch += 1.0;
    }
    red[0][threadIdx.x] = es;
    red[1][threadIdx.x] = ec;
    red[2][threadIdx.x] = er;
    red[3][threadIdx.x] = zero_mismatch;
    __syncthreads();
    for (int h = FGB_THREADS / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) {
            for (int q = 0; q < 3; ++q) red[q][threadIdx.x] = fmax(red[q][threadIdx.x], red[q][threadIdx.x + h]);
            red[3][threadIdx.x] += red[3][threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x < 4) out[4 * blockIdx.x + threadIdx.x] = red[threadIdx.x][0];
}

static void fastgen_bounds(double measured[4], double assumed[2], hipStream_t stream) {
    RBX_REQUIRE(measured != nullptr && assumed != nullptr);
    double *dev_out = (double *)scratch(SCRATCH_SMALL, (size_t)FGB_BLOCKS * 4 * sizeof(double), stream);
    hipLaunchKernelGGL(fastgen_bounds_kernel, dim3(FGB_BLOCKS), dim3(FGB_THREADS), 0, stream, dev_out);
    RBX_HIP(hipGetLastError());
    std::vector<double> h((size_t)FGB_BLOCKS * 4);
    RBX_HIP(hipMemcpyAsync(h.data(), dev_out, h.size() * sizeof(double), hipMemcpyDeviceToHost, stream));
    RBX_HIP(hipStreamSynchronize(stream));
    for (int q = 0; q < 4; ++q) measured[q] = 0.0;
    for (int b = 0; b < FGB_BLOCKS; ++b) {
        for (int q = 0; q < 3; ++q) measured[q] = fmax(measured[q], h[4 * b + q]);
        measured[3] += h[4 * b + 3];
    }
    assumed[0] = (double)BM_ES;
    assumed[1] = (double)BM_ER;
}

}  // namespace rbx

using namespace rbx;

extern "C" rbx_status rbx_slskge3_bf16split(char layout, char opS, char opA, int64_t d, int64_t n, int64_t m,
                                            float alpha, const rbx_dense_skop *S, int64_t ro_s, int64_t co_s,
                                            const float *A, int64_t lda, float beta, float *B, int64_t ldb,
                                            int n_terms, void *stream) {
    RBX_API_BEGIN
    bf16_split_sketch(layout, opS, opA, d, n, m, alpha, S, ro_s, co_s, A, lda, beta, B, ldb, n_terms,
                      (hipStream_t)stream);
    RBX_API_END
}

extern "C" rbx_status rbx_bf16_fastgen_bounds(double *measured, double *assumed, void *stream) {
    RBX_API_BEGIN
    fastgen_bounds(measured, assumed, (hipStream_t)stream);
    RBX_API_END
}
