// rbx_wide.hip -- plans and launches the fused dense sketches (rbx_wide.hh): the tile width and the K ranges, the reduction of
// the ranges' partials.
#include <algorithm>
#include <type_traits>

#include "rbx_wide.hh"

namespace rbx {

// C[i, j] = alpha * sum_s part[s][i * ldp + j] + beta * C[i, j], FP64 sums in a
// fixed order; column N - 1 of C apart at xC when given.  A workgroup takes a
// TR x 4 TQ tile; G threads per four columns sum the splits s = g, g + G, ...,
// then the G sums are added in order (G > 1 when the output alone has too few
// entries to keep the loads of many splits in flight).  Tiles with one thread
// per quad are 8 x 128, 512-byte (FP32) runs of every partial.
template <typename T, int G>
__global__ __launch_bounds__(256) void wide_reduce_kernel(const T *part, int nS, int64_t M, int64_t N, int64_t ldp,
                                                          double alpha, double beta, T *C, int64_t crs, int64_t ccs,
                                                          T *xC, int64_t xcrs) {
    constexpr int TR = G == 1 ? 8 : 4, TQ = 256 / G / TR, TC = 4 * TQ;
    __shared__ double sums[G][TR][TC + 1];
    typedef T t4 __attribute__((ext_vector_type(4)));
    const int64_t ntc = (N + TC - 1) / TC;
    const int64_t i0 = (int64_t)(blockIdx.x / ntc) * TR, j0 = (int64_t)(blockIdx.x % ntc) * TC;
    const int tid = threadIdx.x;
    {
        const int c4 = 4 * (tid % TQ), r = (tid / TQ) % TR, gq = tid / (TQ * TR);
        const int64_t i = i0 + r, j = j0 + c4, total = M * ldp;
        double v[4] = {0.0, 0.0, 0.0, 0.0};
        if (i < M && j < ldp) {
            const T *p = part + i * ldp + j;
            int s = gq;
            for (; s + 7 * G < nS; s += 8 * G) {
                t4 x[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) x[u] = *(const t4 *)(p + (int64_t)(s + u * G) * total);
#pragma unroll
                for (int u = 0; u < 8; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] += (double)x[u][e];
            }
            for (; s < nS; s += G) {
                const t4 x = *(const t4 *)(p + (int64_t)s * total);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += (double)x[e];
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) sums[gq][r][c4 + e] = v[e];
    }
    __syncthreads();
    const bool cm = crs == 1;  // consecutive threads along C's unit stride
    for (int e = tid; e < TR * TC; e += 256) {
        const int ti = cm ? e % TR : e / TC, tj = cm ? e / TR : e % TC;
        const int64_t i = i0 + ti, j = j0 + tj;
        if (i < M && j < N) {
            double v = sums[0][ti][tj];
#pragma unroll
            for (int q = 1; q < G; ++q) v += sums[q][ti][tj];
            T *c = (xC != nullptr && j == N - 1) ? xC + i * xcrs : C + i * crs + j * ccs;
            double out = alpha * v;
            if (beta != 0.0) out += beta * (double)(*c);
            *c = (T)out;
        }
    }
}

// The tail's outputs: out[j][i * ors[j]] = alpha * (sum over splits of
// tpart[(s * nt + j) * Mt + mo + i]) + beta * out, FP64 sums.  G threads per
// output entry: G = 1 sums the splits in order; G = 64 (many splits) has lane
// l sum splits l, l + 64, ..., then a butterfly (a fixed order).
template <typename T, int G>
__global__ __launch_bounds__(256) void wide_tail_reduce_kernel(const T *tpart, int nS, int64_t M, int64_t Mt, int mo,
                                                               TailCols<T> tc, double alpha, double beta) {
    const int nt = tc.nt;
    const int g = threadIdx.x % G;
    const int64_t e = (int64_t)blockIdx.x * (256 / G) + threadIdx.x / G;
    if (e >= M * nt) return;  // uniform per group
    const int64_t i = e % M;
    const int j = (int)(e / M);
    double v = 0.0;
    for (int s = g; s < nS; s += G) v += (double)tpart[((int64_t)s * nt + j) * Mt + mo + i];
    if constexpr (G == 64) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
        if (g != 0) return;
    }
    T *c = nullptr;
    int64_t rs = 0;
#pragma unroll
    for (int q = 0; q < WIDE_TAIL; ++q)
        if (q == j) {
            c = tc.out[q];
            rs = tc.ors[q];
        }
    c += i * rs;
    double out = alpha * v;
    if (beta != 0.0) out += beta * (double)(*c);
    *c = (T)out;
}

// Y (K < 4 rows) as four rows, the rest zeros, unit stride along K
template <typename T>
__global__ __launch_bounds__(256) void pad_k4_kernel(const T *D, int64_t drs, int64_t dcs, int K, int64_t N, T *out) {
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < 4 * N; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = e / 4;
        const int k = (int)(e % 4);
        out[e] = k < K ? D[k * drs + j * dcs] : (T)0;
    }
}

// Scratch, or nullptr when the device cannot provide it.
static void *try_scratch(size_t bytes, hipStream_t stream) {
    try {
        return scratch(SCRATCH_SPLITK, bytes, stream);
    } catch (const Fail &f) {
        if (f.st != RBX_OUT_OF_MEMORY) throw;
        clear_error();
        return nullptr;
    }
}

// Tile width, tail columns and K ranges of one product.  The time of a
// workgroup's 32-deep chunk is its MFMAs (64 x tile x 32 at the matrix rate,
// also for columns that do not exist) plus the operator's generation (2048
// entries, the same for every tile width); rounds of one workgroup per CU.
// More K ranges fill the chip, but their partials are written and read.
struct WidePlan {
    int tile, tw, nS;
    int64_t kw;
};
constexpr size_t WIDE_PART_MAX = 16ull << 30;  // partials above this: fewer ranges

template <typename T>
static WidePlan wide_plan(const GemmProblem &pb, int ko, int mo, bool NU, bool split_ok) {
    constexpr bool F64 = sizeof(T) == 8;
    // clocks of a CU: 2048 Gaussian entries (measured: 1.2 a clock), chunk overhead,
    // a workgroup's start and end
    const double gen = pb.g.gauss ? 1700.0 : 800.0, over = 300.0, fixed = 5000.0, mhz = 2100.0;
    const double flop_clk = F64 ? 128.0 : 256.0;
    // FP32 sums are kept in ranges of at most 4096 terms, FP64 needs no bound
    const int64_t kw_max = F64 ? 16384 : 4096;
    const int64_t Kp = pb.K + ko, chunks = (Kp + WD_KC - 1) / WD_KC;
    const int64_t nMB = (pb.M + mo + WD_MT - 1) / WD_MT;
    const int cus = num_cus();
    // columns, waves along the rows, blocks per wave (wide_launch_tile)
    static const struct { int cols, wm, cb; } tiles[] = {
        {32, 4, 1},  {64, 2, 1},  {128, 1, 1}, {192, 2, 3}, {256, 1, 2}, {320, 2, 5},
        {384, 1, 3}, {448, 2, 7}, {512, 1, 4}, {640, 1, 5}, {768, 1, 6}, {1024, 1, 8}};
    WidePlan best{};
    double best_t = 1e300;
    for (const auto &tl : tiles) {
        const int tile = tl.cols;
        if (F64 && tile > 512) break;
        // (FP32, unit stride along N) the 1024-wide form has too few registers
        if (NU && tile == 1024) break;
        if (NU && pb.N < tl.cb) continue;
        // two waves read the same columns: only where one tile is the whole
        // output (100000 columns, K = 2000, FP32: 448 wide 630 us, 512 wide 590)
        if (tl.wm == 2 && tile > 64 && pb.N > tile) continue;
        const bool two = wide_waves<T>(tl.wm, tl.cb, 0) == 4;  // two workgroups per CU
        for (int tail = 0; tail < 2; ++tail) {
            int tw = 0;
            if (tail) {
                tw = (int)std::min<int64_t>(pb.N - tile, WIDE_TAIL + 1);
                if (NU || !split_ok || (tile != 128 && tile != 256) || tw < 1 || tw > WIDE_TAIL) continue;
            }
            const int64_t nNB = tail ? 1 : (pb.N + tile - 1) / tile;
            const int64_t wgs = nMB * nNB;
            const double chunk_clk = 64.0 * tile * 64.0 / flop_clk + gen + over + (tw > 1 ? 400.0 : 100.0 * tw);
            const int64_t ns_min = split_ok ? (Kp + kw_max - 1) / kw_max : 1;
            for (int r = 0; r <= 8; ++r) {
                int64_t ns = r == 0 ? ns_min : std::max<int64_t>(ns_min, r * (int64_t)cus / wgs);
                if (!split_ok) ns = 1;
                if (ns < 1) ns = 1;
                const int64_t cps = (chunks + ns - 1) / ns;  // chunks per range
                ns = (chunks + cps - 1) / cps;
                const double part = (double)ns * (double)pb.M * (double)pb.N * sizeof(T);
                if (ns > 1 && part > (double)WIDE_PART_MAX) continue;
                // with two workgroups on a CU the last round overlaps the one before
                double rounds = (double)((wgs * ns + cus - 1) / cus);
                if (two && rounds > 1) rounds = std::min(rounds, (double)(wgs * ns) / cus + 0.5);
                double t = rounds * (cps * chunk_clk + fixed) / mhz;
                if (ns > 1) t += 5.0 + 2.0 * part / 3.5e6;
                if (tail) t += 3.0;
                if (t < best_t) {
                    best_t = t;
                    best = WidePlan{tile, tw, (int)ns, cps * WD_KC};
                }
            }
        }
    }
    if (best.tile == 0) {  // partials too large for any number of ranges
        const int tile = pb.N < 512 ? 128 : 512;
        best = WidePlan{tile, 0, 1, chunks * WD_KC};
    }
    return best;
}

template <typename T>
void wide_run(const GemmProblem &pb, hipStream_t stream) {
    RBX_REQUIRE(pb.gen_is_x && pb.M > 0 && pb.N > 0 && pb.K > 0);
    WideProblem<T> w{};
    w.M = pb.M;
    w.N = pb.N;
    w.K = pb.K;
    w.g = pb.g;
    const int off = (int)(pb.g.b_off & 3);
    w.g.b_off -= off;
    const bool rows = pb.g.b_along_rows != 0;
    w.mo = rows ? off : 0;
    w.ko = rows ? 0 : off;
    if (pb.sbuf != nullptr) {
        w.S = (const T *)pb.sbuf + pb.soff;
        w.srs = pb.srs;
        w.scs = pb.scs;
    }
    w.D = (const T *)pb.D;
    w.drs = pb.drs;
    w.dcs = pb.dcs;
    w.xD = (const T *)pb.xD;
    w.C = (T *)pb.C;
    w.crs = pb.crs;
    w.ccs = pb.ccs;
    w.xC = (T *)pb.xC;
    w.xcrs = pb.xcrs;
    w.alpha = (T)pb.alpha;
    w.beta = (T)pb.beta;
    if (pb.K < 4 || (pb.drs != 1 && pb.dcs != 1)) {
        RBX_REQUIRE(pb.K < 4 && pb.xD == nullptr && pb.xC == nullptr);
        T *pad = (T *)scratch(SCRATCH_BF16, (size_t)safe_mul(pb.N, 4) * sizeof(T), stream);
        const unsigned blocks = (unsigned)std::min<int64_t>((pb.N + 63) / 64, 65536);
        hipLaunchKernelGGL(pad_k4_kernel<T>, dim3(blocks), dim3(256), 0, stream, w.D, pb.drs, pb.dcs, (int)pb.K, pb.N,
                           pad);
        RBX_HIP(hipGetLastError());
        w.D = pad;
        w.K = 4;
        w.drs = 1;
        w.dcs = 4;
    }
    const bool NU = w.drs != 1;
    RBX_REQUIRE(!NU || pb.xD == nullptr);
    GemmProblem sized = pb;
    sized.K = w.K;
    WidePlan p = wide_plan<T>(sized, w.ko, w.mo, NU, true);
    w.nMB = (int)((pb.M + w.mo + WD_MT - 1) / WD_MT);
    const int64_t Mt = 64 * (int64_t)w.nMB;
    char *ws = nullptr;
    size_t part_bytes = 0;
    if (p.nS > 1 || p.tw > 0) {
        w.ldp = (pb.N - p.tw + 3) / 4 * 4;
        if (p.nS > 1) part_bytes = ((size_t)p.nS * pb.M * w.ldp * sizeof(T) + 255) / 256 * 256;
        ws = (char *)try_scratch(part_bytes + (size_t)p.nS * p.tw * Mt * sizeof(T), stream);
        if (ws == nullptr) p = wide_plan<T>(sized, w.ko, w.mo, NU, false);
    }
    w.nS = p.nS;
    w.kw = p.kw;
    w.N = pb.N - p.tw;
    w.nNB = (int)((w.N + p.tile - 1) / p.tile);
    RBX_REQUIRE((int64_t)w.nMB * w.nNB < (1ll << 31) / w.nS);
    if (p.nS > 1) w.part = (T *)ws;
    if (p.tw > 0) {
        w.tpart = (T *)(ws + part_bytes);
        w.tc.nt = p.tw;
        for (int j = 0; j < WIDE_TAIL; ++j) {  // unused slots repeat the last column (loaded, never written)
            const int64_t c = w.N + std::min(j, p.tw - 1);
            const bool last = c == pb.N - 1;
            w.tc.col[j] = (last && pb.xD) ? (const T *)pb.xD : w.D + c * w.dcs;
            w.tc.rs[j] = (last && pb.xD) ? pb.xdrs : w.drs;
            w.tc.out[j] = (last && pb.xC) ? (T *)pb.xC : w.C + c * w.ccs;
            w.tc.ors[j] = (last && pb.xC) ? pb.xcrs : w.crs;
        }
        w.xD = nullptr;  // the last column is the tail's
        w.xC = nullptr;
    } else {
        for (int j = 0; j < WIDE_TAIL; ++j) w.tc.col[j] = w.D;
    }
    const bool gauss = pb.g.gauss != 0;
    {
        ProfScope prof(sizeof(T) == 8 ? "f64_wide_kernel" : "f32_wide_kernel", stream);
        if (w.S != nullptr && w.srs == 1) wide_launch<T, WIDE_MEM, true>(NU, p.tile, p.tw, w, stream);
        else if (w.S != nullptr) wide_launch<T, WIDE_MEM, false>(NU, p.tile, p.tw, w, stream);
        else if (gauss && rows) wide_launch<T, WIDE_GAUSS, true>(NU, p.tile, p.tw, w, stream);
        else if (gauss) wide_launch<T, WIDE_GAUSS, false>(NU, p.tile, p.tw, w, stream);
        else if (rows) wide_launch<T, WIDE_UNIFORM, true>(NU, p.tile, p.tw, w, stream);
        else wide_launch<T, WIDE_UNIFORM, false>(NU, p.tile, p.tw, w, stream);
        RBX_HIP(hipGetLastError());
    }
    if (w.nS > 1) {
        ProfScope prof(sizeof(T) == 8 ? "f64_reduce_kernel" : "f32_reduce_kernel", stream);
        auto go = [&](auto gv) {
            constexpr int G = decltype(gv)::value, TR = G == 1 ? 8 : 4, TC = 4 * (256 / G / TR);
            const int64_t nt = ((w.M + TR - 1) / TR) * ((w.N + TC - 1) / TC);
            RBX_REQUIRE(nt < (1ll << 31));
            hipLaunchKernelGGL((wide_reduce_kernel<T, G>), dim3((unsigned)nt), dim3(256), 0, stream, (const T *)w.part,
                               w.nS, w.M, w.N, w.ldp, pb.alpha, pb.beta, w.C, w.crs, w.ccs, w.xC, w.xcrs);
        };
        // enough threads for about 16 waves per CU, at most one per 4 splits
        const int64_t quads = w.M * w.ldp / 4, want = 256 * 1024;
        if (quads >= want || w.nS < 8) go(std::integral_constant<int, 1>{});
        else if (quads * 4 >= want || w.nS < 32) go(std::integral_constant<int, 4>{});
        else go(std::integral_constant<int, 16>{});
        RBX_HIP(hipGetLastError());
    }
    if (p.tw > 0) {
        const int64_t n = w.M * p.tw;
        if (w.nS <= 16)
            hipLaunchKernelGGL((wide_tail_reduce_kernel<T, 1>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                               (const T *)w.tpart, w.nS, w.M, Mt, w.mo, w.tc, pb.alpha, pb.beta);
        else
            hipLaunchKernelGGL((wide_tail_reduce_kernel<T, 64>), dim3((unsigned)((n + 3) / 4)), dim3(256), 0, stream,
                               (const T *)w.tpart, w.nS, w.M, Mt, w.mo, w.tc, pb.alpha, pb.beta);
        RBX_HIP(hipGetLastError());
    }
}
template void wide_run<float>(const GemmProblem &, hipStream_t);
template void wide_run<double>(const GemmProblem &, hipStream_t);

}  // namespace rbx
