// rbx_wide.hh -- fused dense sketches, FP64 and FP32:
//     C[M x N] = alpha * G[M x K] * Y[K x N] + beta * C
// G the operator, generated from its Philox counters (or read from memory
// when it is materialised), Y the dense operand (either unit stride), any
// sizes and any submatrix of the operator.
//
// One 512-thread workgroup per 64 x NT output tile, or per share of such a tile's
// K (WideWork).  Every 32-deep chunk of the tile's operator rows is generated
// once into LDS (each thread one counter, four entries) while the chunk before it
// is multiplied: waves 0-3 generate before their MFMAs, waves 4-7 after, so the
// two waves that share a SIMD are in opposite phases.  The 8 waves form a WM x 8
// / WM grid; each owns RB x CB blocks of v_mfma_f{64,32}_16x16x4 (WM * RB = 4, NT
// = 128 CB / WM).  The dense operand goes straight from memory into the MFMA
// registers, one 16-deep step ahead of its use: lane (g = l / 16, c = l % 16)
// holds k = 4 g .. 4 g + 3 of its columns, so with unit stride along K a
// column's 16 k are one run of four lanes' vectors, and with unit stride along
// N a lane holds CB neighbouring columns of four rows.
//
// What bounds it: the SIMDs' issue, shared by the MFMAs and the generator (FP64
// 2048 x 131072 x 1000: 6.8 ms of MFMAs at the peak rate, 8.1 ms measured), and
// how evenly the tiles fill the CUs.  Several columns of tiles need the same
// operator rows: generated once ahead (WIDE_PRE) instead of once in each, FP64
// 1032 x 34498 x 1189 takes 1572 us instead of 1716.  A last round of few tiles
// is shared out instead of leaving CUs idle: FP32 50001 x 777 x 301 (782 tiles on
// 256 CUs) 392 -> 335 us; with both, the FP32 right sketch 100000 x 2000 to 110
// columns 568 -> 469 us.
//
// Sizes that do not fit: K (at least 4) is rounded up to whole chunks, the
// dense values past it are zeros (the operator's are whatever the counters
// give); rows and
// columns past the edge read the edge again and are not stored.  An operator
// window that starts inside a counter (b_off % 4 != 0) is moved back to the
// counter's start: ko extra k with zero dense values, or mo extra rows that
// are not stored.
#pragma once
#include <type_traits>

#include "rbx_gemm_common.hh"

namespace rbx {

constexpr int WD_THR = 512, WD_MT = 64, WD_KC = 32;

template <typename T>
struct WideMma;
template <>
struct WideMma<double> {
    typedef double acc_t __attribute__((ext_vector_type(4)));
    static constexpr int LDK = 34;  // row stride 68 words: 16 rows' 16-byte reads cover the banks once
    static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // The LDS row of a tile's row: the results r of lane l are the MFMA's rows
    // l / 16 + 4 r, which with this order (4 x 4 within 16 rows, transposed) are
    // the tile's rows 4 (l / 16) + r, as FP32's are.
    static __device__ __forceinline__ int lds_row(int y) { return (y & ~15) | 4 * (y & 3) | ((y >> 2) & 3); }
};
template <>
struct WideMma<float> {
    typedef float acc_t __attribute__((ext_vector_type(4)));
    static constexpr int LDK = 36;
    static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int lds_row(int y) { return y; }
};

// Tail columns: up to WIDE_TAIL output columns past the last whole tile (the
// right-hand side of [A b]) are formed by the threads that generate the
// operator, from the four entries each holds per chunk, with VALU FMAs.  The
// generator of operator rows along K holds one row's four consecutive k (one
// accumulator per column); the one of counters along the rows holds four rows
// at one k (four per column).  The dense values of chunk c + 1 are loaded
// right after chunk c's are used, so they have a chunk's MFMAs to arrive.  TW
// columns are always loaded and accumulated (TW = 1, or 4 with the unused
// ones repeating the last real column), so the chunk loop has no branch.
constexpr int WIDE_TAIL = 4;
// Dense column j's element k at col[j][k * rs[j]], its output's element i at
// out[j][i * ors[j]]; entries nt .. WIDE_TAIL - 1 of col / rs repeat nt - 1.
template <typename T>
struct TailCols {
    const T *col[WIDE_TAIL];
    int64_t rs[WIDE_TAIL];
    T *out[WIDE_TAIL];
    int64_t ors[WIDE_TAIL];
    int nt;
};
template <typename T, bool ROWS, int TW>
struct WideTail {
    static constexpr int R = ROWS ? 4 : 1;  // output rows per thread
    static constexpr int E = ROWS ? 1 : 4;  // dense values per column per chunk
    T acc[TW][R];
    T cur[TW][E];  // the dense values of the chunk being generated

    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int j = 0; j < TW; ++j)
#pragma unroll
            for (int r = 0; r < R; ++r) acc[j][r] = (T)0;
    }
    // cur = dense values of k .. k + E - 1, zeros outside [0, K)
    __device__ __forceinline__ void load(const TailCols<T> &tc, int64_t k, int64_t K) {
#pragma unroll
        for (int j = 0; j < TW; ++j)
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int64_t q = k + e, in = q < 0 ? 0 : (q < K ? q : K - 1);
                const T v = tc.col[j][in * tc.rs[j]];
                cur[j][e] = in == q ? v : (T)0;
            }
    }
    __device__ __forceinline__ void step(const T (&ent)[4]) {
#pragma unroll
        for (int j = 0; j < TW; ++j) {
            if constexpr (ROWS) {
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[j][r] = fma(ent[r], cur[j][0], acc[j][r]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[j][0] = fma(ent[e], cur[j][e], acc[j][0]);
            }
        }
    }
    // The workgroup's 64 x nt partial into out[j * Mt + row].  Rows along K:
    // the eight threads of a row are adjacent lanes (butterfly).  Counters
    // along the rows: lanes l, l ^ 16, l ^ 32, l ^ 48 of a wave share rows
    // (butterfly), then the eight waves are summed in order through `red`
    // (8 * TW * 64 values).  Every thread calls this (it has a barrier).
    __device__ __forceinline__ void finish(int nt, int tid, int frow, int fcell, T *red, T *out, int64_t Mt) {
        const int lane = tid & 63, wave = tid >> 6;
        if constexpr (!ROWS) {
#pragma unroll
            for (int j = 0; j < TW; ++j) {
                T v = acc[j][0];
                v += __shfl_xor(v, 1);
                v += __shfl_xor(v, 2);
                v += __shfl_xor(v, 4);
                if (j < nt && fcell == 0) out[j * Mt + frow] = v;
            }
        } else {
#pragma unroll
            for (int j = 0; j < TW; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    T v = acc[j][r];
                    v += __shfl_xor(v, 16);
                    v += __shfl_xor(v, 32);
                    if (lane < 16) red[(wave * TW + j) * 64 + frow + r] = v;
                }
            __syncthreads();
            if (tid < 64 * nt) {
                const int j = tid >> 6, row = tid & 63;
                T v = red[j * 64 + row];
#pragma unroll
                for (int w = 1; w < WD_THR / 64; ++w) v += red[(w * TW + j) * 64 + row];
                out[j * Mt + row] = v;
            }
        }
    }
};

// How the 64 x tile output tiles and their chunks (32 k each, `chunks` per tile)
// go to workgroups: the first `whole` tiles to one each, each of the `rest` tiles
// after them to `each`, all of which do the same share of the chunks; the i-th
// of tile v writes its sums to the slot v * each + i.
struct WideWork {
    int whole, rest, each, nMB, chunks;
    int q, r;  // chunks = q * each + r

    __host__ __device__ int first(int i) const { return i * q + (i < r ? i : r); }
};

template <typename T>
struct WideProblem {
    int64_t M, N, K;       // N without the tail columns
    GenMap g;              // b_off a multiple of 4
    const T *S;            // materialised operator: element (i, k) at S[i * srs + k * scs]
    int64_t srs, scs;
    const float *pre;      // WIDE_PRE: the operator's chunks (wide_pre_kernel)
    T scale;               // and its entries' scale
    int ko, mo;            // extra k / rows in front (see above); one of them is 0
    const T *D;
    int64_t drs, dcs;
    const T *xD;           // column N - 1 (unit stride) when not null
    T *C, *xC;
    int64_t crs, ccs, xcrs;
    T alpha, beta;
    WideWork wk;
    T *part;               // partials, one 64 x tile block per slot, rows along C's unit stride
    int part_cols;         // 1: columns are contiguous (element (i, j) at i * tile + j), 0: rows (i + 64 j)
    TailCols<T> tc;        // tail columns, partials at tpart[(slot * tc.nt + j) * 64 + row]
    T *tpart;
};

template <typename T, int N>
struct WideVec {
    typedef T type __attribute__((ext_vector_type(N), aligned(sizeof(T))));
};

// Waves per SIMD that the registers are bounded for: two workgroups per CU
// where the accumulators leave room (the last round of a grid then ends sooner,
// and one workgroup's barrier is the other's work).  (FP32, unit stride along N:
// 384 columns spill at 128 registers.)
template <typename T>
constexpr int wide_waves(bool NU, int WM, int CB, int TW) {
    const int acc = 4 / WM * CB * (int)sizeof(T) + (NU && sizeof(T) == 4 ? 8 : 0);
    if (acc <= 8 && TW == 0) return 8;  // 32 columns: four workgroups (FP64 at three: 2% slower)
    return acc + 4 * TW * (int)sizeof(T) / 4 <= 48 ? 4 : 2;
}

// The operator: uniform or Gaussian, generated here, read from memory, or
// generated ahead of this kernel chunk by chunk (WIDE_PRE, with ROWS = false
// for either direction).  ROWS: its counters (or its unit stride) run along the
// output's rows, else along K.
enum WideOp { WIDE_UNIFORM = 0, WIDE_GAUSS = 1, WIDE_MEM = 2, WIDE_PRE = 3 };

// NU: the dense operand's unit stride runs along N (else along K).
template <typename T, int OP, bool ROWS, bool NU, int WM, int CB, int TW>
__global__ __launch_bounds__(WD_THR, OP == WIDE_MEM ? (wide_waves<T>(NU, WM, CB, TW) == 2 ? 2 : 4)
                                                     : wide_waves<T>(NU, WM, CB, TW)) void wide_kernel(const WideProblem<T> pb) {
    using MM = WideMma<T>;
    constexpr int RB = 4 / WM, WN = 8 / WM, LDK = MM::LDK;
    constexpr int NT = 16 * CB * WN;
    constexpr int RED = TW > 0 ? 8 * TW * 64 : 0;
    constexpr int LDS_N = 2 * WD_MT * LDK > RED ? 2 * WD_MT * LDK : RED;
    __shared__ __attribute__((aligned(16))) T Ss[LDS_N];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int lc = lane & 15, lg = lane >> 4;

    // ---- this workgroup's chunks c0 .. c0 + nchunks - 1 of tile t.  XCD-aware
    // order: consecutive tiles (same chunks and columns, so the same dense
    // operand) on one XCD
    const WideWork wk = pb.wk;
    auto xcd_order = [](int b, int n) {
        const int xcd = b % 8, xi = b / 8;
        return xcd * (n / 8) + (xcd < n % 8 ? xcd : n % 8) + xi;
    };
    int t, c0 = 0, nchunks = wk.chunks, slot = -1;
    if ((int)blockIdx.x < wk.whole) {
        t = xcd_order(blockIdx.x, wk.whole);
    } else {
        const int o = xcd_order(blockIdx.x - wk.whole, wk.rest * wk.each), i = o / wk.rest, v = o - i * wk.rest;
        t = wk.whole + v;
        c0 = wk.first(i);
        nchunks = wk.first(i + 1) - c0;
        slot = v * wk.each + i;
    }
    const int nb = t / wk.nMB, mb = t - nb * wk.nMB;
    const int64_t m0 = (int64_t)mb * WD_MT, n0 = (int64_t)nb * NT;
    const int64_t kbeg = (int64_t)c0 * WD_KC;
    const int64_t Kp = pb.K + pb.ko;
    const GenMap g = pb.g;
    constexpr bool GAUSS = OP == WIDE_GAUSS;

    typename MM::acc_t acc[RB][CB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[i][j] = typename MM::acc_t{0, 0, 0, 0};

    // ---- operator chunk: rows along K (!ROWS): the thread owns cell tid % 8
    // of LDS row tid / 8; counters along the rows (ROWS): rows 4 (tid % 16) .. + 3
    // of column tid / 16.  Row r, k at Ss[lds_row(r) * LDK + k].
    const int frow = ROWS ? 4 * (tid & 15) : MM::lds_row(tid >> 3), fcell = ROWS ? tid >> 4 : tid & 7;
    uint64_t foff = ROWS ? (uint64_t)((g.a_off + kbeg + fcell) * g.P + ((g.b_off + m0) >> 2) + (tid & 15))
                               : (uint64_t)((g.a_off + m0 + frow) * g.P + ((g.b_off + kbeg) >> 2) + fcell);
    const uint64_t fstep = ROWS ? WD_KC * (uint64_t)g.P : WD_KC / 4;  // counters per chunk
    WideTail<T, ROWS, TW == 0 ? 1 : TW> tl;
    const int64_t tk = kbeg - pb.ko + (ROWS ? fcell : 4 * fcell);  // the thread's first k of chunk 0
    if constexpr (TW > 0) {
        tl.zero();
        tl.load(pb.tc, tk, pb.K);
    }
    // a materialised operator's entries of the next chunk, loaded a chunk ahead
    T mem[4];
    auto load_op = [&](int c) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int64_t r = m0 + frow + (ROWS ? e : 0) - pb.mo;
            const int64_t k = kbeg - pb.ko + WD_KC * (int64_t)c + (ROWS ? fcell : 4 * fcell + e);
            const int64_t ri = r < 0 ? 0 : (r < pb.M ? r : pb.M - 1), ki = k < 0 ? 0 : (k < pb.K ? k : pb.K - 1);
            const T v = pb.S[ri * pb.srs + ki * pb.scs];
            mem[e] = ri == r && ki == k ? v : (T)0;
        }
    };
    typedef float f4 __attribute__((ext_vector_type(4)));
    f4 pre4;
    const float *prep = nullptr;
    if constexpr (OP == WIDE_PRE) {
        prep = pb.pre + ((int64_t)mb * wk.chunks + c0) * (WD_MT * WD_KC) + frow * WD_KC + 4 * fcell;
        pre4 = *(const f4 *)prep;
    }
    if constexpr (OP == WIDE_MEM) load_op(0);
    auto gen_chunk = [&](int c, T *lds) {
        T ent[4];
        if constexpr (OP == WIDE_MEM) {
#pragma unroll
            for (int e = 0; e < 4; ++e) ent[e] = mem[e];
        } else if constexpr (OP == WIDE_PRE) {
#pragma unroll
            for (int e = 0; e < 4; ++e) ent[e] = (T)pre4[e] * pb.scale;
        } else {
            const float4 v = gen4(GAUSS, ctr_add(g.ctr, foff), g.k0, g.k1);
            foff += fstep;  // (the chunks are generated in order)
            ent[0] = entry_value<T>(v.x, GAUSS);
            ent[1] = entry_value<T>(v.y, GAUSS);
            ent[2] = entry_value<T>(v.z, GAUSS);
            ent[3] = entry_value<T>(v.w, GAUSS);
        }
        if constexpr (ROWS) {
#pragma unroll
            for (int e = 0; e < 4; ++e) lds[MM::lds_row(frow + e) * LDK + fcell] = ent[e];
        } else {
            T *row = lds + (tid >> 3) * LDK + 4 * fcell;  // row lds_row(frow)
#pragma unroll
            for (int e = 0; e < 4; ++e) row[e] = ent[e];
        }
        if constexpr (OP == WIDE_MEM) load_op(c + 1);
        if constexpr (OP == WIDE_PRE) {  // (one chunk past a tile's last is inside the buffer)
            prep += WD_MT * WD_KC;
            pre4 = *(const f4 *)prep;
        }
        if constexpr (TW > 0) {
            tl.step(ent);
            tl.load(pb.tc, tk + WD_KC * (int64_t)(c + 1), pb.K);  // the next chunk's
        }
    };

    // ---- dense operand of one 16-deep step, b[j][q] = Y[16 s + 4 lg + q - ko][column j]
    const int64_t wcol = n0 + wn * (16 * CB);
    T b[CB][4];
    const T *colp[NU ? 1 : CB];   // !NU: column j's element k = 4 lg - ko; NU: column cs of that row
    int64_t cs = wcol + CB * lc;  // NU: the lane's first column, moved back inside the matrix
    if constexpr (NU) {
        if (cs > pb.N - CB) cs = pb.N - CB;
        colp[0] = pb.D + cs;
    } else {
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            int64_t col = wcol + 16 * j + lc;
            if (col > pb.N - 1) col = pb.N - 1;
            colp[j] = (pb.xD != nullptr && col == pb.N - 1) ? pb.xD : pb.D + col * pb.dcs;
        }
    }
    const int64_t k_lane = 4 * lg - pb.ko;
    auto is_edge = [&](int64_t s) { return 16 * s < pb.ko || 16 * s + 16 > Kp; };
    // Addresses of a step's loads: element offset of the lane's four k (!NU)
    // or of row q (NU), inside the matrix also at the ends of K.
    int64_t koff, roff[NU ? 4 : 1];
    auto address = [&](int64_t s) {
        const int64_t k = 16 * s + k_lane;
        if constexpr (NU) {
#pragma unroll
            for (int q = 0; q < 4; ++q) roff[q] = (k + q) * pb.drs;
            if (is_edge(s)) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int64_t kq = k + q < 0 ? 0 : (k + q < pb.K ? k + q : pb.K - 1);
                    roff[q] = kq * pb.drs;
                }
            }
        } else {
            koff = k < 0 ? 0 : (k < pb.K - 4 ? k : pb.K - 4);
        }
    };
    auto load_col = [&](int j) {
        const typename WideVec<T, 4>::type v = *(const typename WideVec<T, 4>::type *)(colp[NU ? 0 : j] + koff);
#pragma unroll
        for (int q = 0; q < 4; ++q) b[j][q] = v[q];
    };
    auto load_row = [&](int q) {
        const T *p = colp[0] + roff[NU ? q : 0];
        // the lane's CB neighbours in one or two loads (of three or four each)
        auto piece = [&](auto j0, auto v) {
            constexpr int J = decltype(j0)::value, V = decltype(v)::value;
            if constexpr (V == 1) {
                b[J][q] = p[J];
            } else {
                const typename WideVec<T, V>::type x = *(const typename WideVec<T, V>::type *)(p + J);
#pragma unroll
                for (int j = 0; j < V; ++j) b[J + j][q] = x[j];
            }
        };
        using std::integral_constant;
        constexpr int V0 = CB <= 4 ? CB : (CB == 5 ? 3 : (CB + 1) / 2);
        piece(integral_constant<int, 0>{}, integral_constant<int, V0>{});
        if constexpr (CB > V0) piece(integral_constant<int, V0>{}, integral_constant<int, CB - V0>{});
    };
    // A step at the ends of K: zeros outside [0, K), and (!NU) the values back
    // in their places where the vector was read from inside the matrix.
    auto fix_edge = [&](int64_t s) {
        const int64_t k = 16 * s + k_lane;
        const int64_t d = NU ? 0 : k - (k < 0 ? 0 : (k < pb.K - 4 ? k : pb.K - 4));
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            T v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                v[q] = (T)0;
                if constexpr (NU) {
                    v[q] = k + q >= 0 && k + q < pb.K ? b[j][q] : (T)0;
                } else {
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (q + d == u) v[q] = b[j][u];
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) b[j][q] = v[q];
        }
    };

    // One step: the operands of step s_next are loaded right after this
    // step's last use of their registers, a whole step ahead (the fence keeps
    // the compiler from moving the loads next to their use).
    auto step = [&](const T *S, int ks, int64_t s, int64_t s_next) {
        if (is_edge(s)) fix_edge(s);
        address(s_next);
        __builtin_amdgcn_s_setprio(1);
        T a[RB][4];
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            const T *src = S + (16 * (RB * wm + i) + lc) * LDK + 16 * ks + 4 * lg;
#pragma unroll
            for (int q = 0; q < 4; ++q) a[i][q] = src[q];
        }
        if constexpr (NU) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
#pragma unroll
                for (int j = 0; j < CB; ++j)
#pragma unroll
                    for (int i = 0; i < RB; ++i) acc[i][j] = MM::mma(a[i][q], b[j][q], acc[i][j]);
                load_row(q);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int j = 0; j < CB; ++j) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int i = 0; i < RB; ++i) acc[i][j] = MM::mma(a[i][q], b[j][q], acc[i][j]);
                load_col(j);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_s_setprio(0);
    };

    const int64_t s_first = kbeg / 16;
    address(s_first);
    if constexpr (NU) {
#pragma unroll
        for (int q = 0; q < 4; ++q) load_row(q);
    } else {
#pragma unroll
        for (int j = 0; j < CB; ++j) load_col(j);
    }

    const bool late = (wave & 4) != 0;
    gen_chunk(0, Ss);
    __syncthreads();
    for (int c = 0; c < nchunks; ++c) {
        const T *S = Ss + (c & 1) * (WD_MT * LDK);
        T *Sn = Ss + ((c + 1) & 1) * (WD_MT * LDK);
        const int64_t s0 = s_first + 2 * c;
        const bool more = c + 1 < nchunks;
        if (more && !late) gen_chunk(c + 1, Sn);
        step(S, 0, s0, s0 + 1);
        step(S, 1, s0 + 1, s0 + 2);
        if (more && late) gen_chunk(c + 1, Sn);
        __syncthreads();
    }

    if constexpr (TW > 0)
        tl.finish(pb.tc.nt, tid, frow, ROWS ? 0 : fcell, Ss,
                  pb.tpart + (int64_t)(slot < 0 ? t : wk.whole + slot) * pb.tc.nt * WD_MT, WD_MT);

    // ---- results: acc[i][j][r] is row 4 lg + r of the i-th 16 rows, column j
    typedef typename WideVec<T, 4>::type vec4;
    if (slot >= 0) {
        T *out = pb.part + (int64_t)slot * (WD_MT * NT);
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            const int row = 16 * (RB * wm + i) + 4 * lg;
            if (m0 + row - pb.mo >= pb.M) continue;
#pragma unroll
            for (int j = 0; j < CB; ++j) {
                // NU: a lane moved back owns only the columns past its neighbour's
                const int64_t gj = NU ? cs + j : wcol + 16 * j + lc;
                if (NU ? gj < wcol + CB * lc : gj >= pb.N) continue;
                const int col = (int)(gj - n0);
                if (pb.part_cols) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) out[(row + r) * NT + col] = acc[i][j][r];
                } else {
                    *(vec4 *)(out + row + col * WD_MT) = vec4{acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
                }
            }
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            const int64_t gi = m0 + 16 * (RB * wm + i) + 4 * lg - pb.mo;
            const int64_t gj = NU ? cs + j : wcol + 16 * j + lc;
            if (NU ? gj < wcol + CB * lc : gj >= pb.N) continue;  // (as above)
            const bool apart = pb.xC != nullptr && gj == pb.N - 1;
            const int64_t rs = apart ? pb.xcrs : pb.crs;
            T *c = (apart ? pb.xC : pb.C + gj * pb.ccs) + gi * rs;
            if (rs == 1 && pb.beta == (T)0 && gi >= 0 && gi + 4 <= pb.M) {
                *(vec4 *)c = vec4{pb.alpha * acc[i][j][0], pb.alpha * acc[i][j][1], pb.alpha * acc[i][j][2],
                                  pb.alpha * acc[i][j][3]};
                continue;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (gi + r < 0 || gi + r >= pb.M) continue;
                T out = pb.alpha * acc[i][j][r];
                if (pb.beta != (T)0) out = out + pb.beta * c[r * rs];
                c[r * rs] = out;
            }
        }
}

// Launches the instantiation of a tile width and a number of tail columns.
template <typename T, int OP, bool ROWS>
void wide_launch(bool nu, int tile, int tw, const WideProblem<T> &pb, hipStream_t st);

template <typename T, int OP, bool ROWS, bool NU, int WM, int CB, int TW>
static void wide_launch_one(const WideProblem<T> &pb, hipStream_t st) {
    hipLaunchKernelGGL((wide_kernel<T, OP, ROWS, NU, WM, CB, TW>), dim3((unsigned)(pb.wk.whole + pb.wk.rest * pb.wk.each)), dim3(WD_THR), 0, st, pb);
}
template <typename T, int OP, bool ROWS, bool NU>
static void wide_launch_tile(int tile, int tw, const WideProblem<T> &pb, hipStream_t st) {
    if constexpr (!NU) {
        if (tw == 1 && tile == 128) return wide_launch_one<T, OP, ROWS, NU, 1, 1, 1>(pb, st);
        if (tw == 1 && tile == 256) return wide_launch_one<T, OP, ROWS, NU, 1, 2, 1>(pb, st);
        if (tw > 1 && tile == 128) return wide_launch_one<T, OP, ROWS, NU, 1, 1, WIDE_TAIL>(pb, st);
        if (tw > 1 && tile == 256) return wide_launch_one<T, OP, ROWS, NU, 1, 2, WIDE_TAIL>(pb, st);
    }
    if (tile == 32) return wide_launch_one<T, OP, ROWS, NU, 4, 1, 0>(pb, st);
    if (tile == 64) return wide_launch_one<T, OP, ROWS, NU, 2, 1, 0>(pb, st);
    if (tile == 128) return wide_launch_one<T, OP, ROWS, NU, 1, 1, 0>(pb, st);
    if (tile == 192) return wide_launch_one<T, OP, ROWS, NU, 2, 3, 0>(pb, st);
    if (tile == 256) return wide_launch_one<T, OP, ROWS, NU, 1, 2, 0>(pb, st);
    if (tile == 320) return wide_launch_one<T, OP, ROWS, NU, 2, 5, 0>(pb, st);
    if (tile == 384) return wide_launch_one<T, OP, ROWS, NU, 1, 3, 0>(pb, st);
    if (tile == 448) return wide_launch_one<T, OP, ROWS, NU, 2, 7, 0>(pb, st);
    if (tile == 512) return wide_launch_one<T, OP, ROWS, NU, 1, 4, 0>(pb, st);
    if constexpr (sizeof(T) == 4) {
        if (tile == 640) return wide_launch_one<T, OP, ROWS, NU, 1, 5, 0>(pb, st);
        if (tile == 768) return wide_launch_one<T, OP, ROWS, NU, 1, 6, 0>(pb, st);
        if constexpr (!NU)
            if (tile == 1024) return wide_launch_one<T, OP, ROWS, NU, 1, 8, 0>(pb, st);
    }
    RBX_FAIL(RBX_UNSUPPORTED, "wide kernels: no tile of %d columns", tile);
}

// One translation unit per (type, operator, orientation) instantiates these.
#define RBX_WIDE_INSTANCES(T, OP, ROWS)                                                                       \
    namespace rbx {                                                                                           \
    template <>                                                                                               \
    void wide_launch<T, OP, ROWS>(bool nu, int tile, int tw, const WideProblem<T> &pb, hipStream_t st) {      \
        if (nu) wide_launch_tile<T, OP, ROWS, true>(tile, tw, pb, st);                                        \
        else wide_launch_tile<T, OP, ROWS, false>(tile, tw, pb, st);                                          \
    }                                                                                                         \
    }

}  // namespace rbx
