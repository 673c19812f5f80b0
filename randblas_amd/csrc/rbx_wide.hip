// rbx_wide.hip -- plans and launches the fused dense sketches (rbx_wide.hh): the
// tile width, how tiles and chunks are shared out, the operator generated ahead,
// the reduction of the shared tiles.
#include <algorithm>
#include <type_traits>

#include "rbx_wide.hh"

namespace rbx {

// The tiles that several workgroups share: C = alpha * (sum of a tile's pieces)
// + beta * C, FP64 sums in a fixed order; column N - 1 of C apart at xC when
// given.  A wave takes 256 consecutive entries of the tile's blocks; NW waves
// share them, wave w summing pieces w, w + NW, ... (NW > 1 when the output alone
// has too few entries to keep the loads of many pieces in flight), and the NW
// sums are added in order.  nsub: sub-blocks of a tile.
template <typename T, int NW>
__global__ __launch_bounds__(NW < 4 ? 256 : 64 * NW) void wide_reduce_kernel(const WideProblem<T> pb, int tile, int nsub,
                                                                             double alpha, double beta) {
    constexpr int WV = NW < 4 ? 4 : NW;
    __shared__ double sums[NW > 1 ? NW : 1][NW > 1 ? 256 : 1];
    typedef T t4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int v = (int)(blockIdx.x / (unsigned)nsub);
    const int sub = (int)(blockIdx.x - (unsigned)v * nsub) * (WV / NW) + (NW > 1 ? 0 : wave);
    const int n = pb.wk.each;
    // the lane's four entries: rows row .. row + 3 of one column, or (part_cols) columns of one row
    const int e0 = 256 * sub + 4 * lane;
    const int row = pb.part_cols ? e0 / tile : e0 % WD_MT, col = pb.part_cols ? e0 - row * tile : e0 / WD_MT;
    const int t = pb.wk.whole + v, nb = t / pb.wk.nMB;
    const int64_t i = (int64_t)(t - nb * pb.wk.nMB) * WD_MT - pb.mo + row, j = (int64_t)nb * tile + col;
    const bool in = e0 < WD_MT * tile && i < pb.M && j < pb.N;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    if (in) {
        const int64_t block = WD_MT * (int64_t)tile;
        const T *p = pb.part + (int64_t)v * n * block + e0;
        for (int u = NW > 1 ? wave : 0; u < n; u += 8 * NW) {
            t4 x[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) x[q] = u + q * NW < n ? *(const t4 *)(p + (u + q * NW) * block) : t4{0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < 8; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] += (double)x[q][e];
        }
    }
    if constexpr (NW > 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) sums[wave][4 * lane + e] = s[e];
        __syncthreads();
        if (wave != 0) return;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s[e] = sums[0][4 * lane + e];
#pragma unroll
            for (int q = 1; q < NW; ++q) s[e] += sums[q][4 * lane + e];
        }
    }
    if (!in) return;
    const bool apart = pb.xC != nullptr && j == pb.N - 1;
    T *c = apart ? pb.xC + i * pb.xcrs : pb.C + i * pb.crs + j * pb.ccs;
    const int64_t cs = pb.part_cols ? pb.ccs : (apart ? pb.xcrs : pb.crs);
    // the entries that exist: e >= lo (rows in front of the first), e < hi
    const int lo = i < 0 ? (int)-i : 0;
    const int64_t left = pb.part_cols ? pb.N - j : pb.M - i;
    const int hi = left < 4 ? (int)left : 4;
    if (cs == 1 && beta == 0.0 && i >= 0 && hi == 4) {
        typedef T u4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
        *(u4 *)c = u4{(T)(alpha * s[0]), (T)(alpha * s[1]), (T)(alpha * s[2]), (T)(alpha * s[3])};
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if ((pb.part_cols ? i < 0 : e < lo) || e >= hi) continue;
        double out = alpha * s[e];
        if (beta != 0.0) out += beta * (double)c[e * cs];
        c[e * cs] = (T)out;
    }
}

// The tail's outputs of one row tile per workgroup: out[j][i * ors[j]] = alpha *
// (sum of the tile's pieces) + beta * out, FP64 sums in a fixed order.  Wave w
// sums pieces w, w + 16, ..., a row per lane.
template <typename T>
__global__ __launch_bounds__(1024) void wide_tail_reduce_kernel(const WideProblem<T> pb, double alpha, double beta) {
    __shared__ double sums[16][WIDE_TAIL][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nt = pb.tc.nt;
    double s[WIDE_TAIL] = {0.0, 0.0, 0.0, 0.0};
    auto add = [&](int slot) {
        const T *p = pb.tpart + (int64_t)slot * nt * WD_MT + lane;
#pragma unroll
        for (int j = 0; j < WIDE_TAIL; ++j)
            if (j < nt) s[j] += (double)p[j * WD_MT];
    };
    const int shared = (int)blockIdx.x - pb.wk.whole;  // which of the shared tiles
    if (shared >= 0) {
        for (int u = wave; u < pb.wk.each; u += 16) add(pb.wk.whole + shared * pb.wk.each + u);
    } else if (wave == 0) {
        add(blockIdx.x);
    }
#pragma unroll
    for (int j = 0; j < WIDE_TAIL; ++j) sums[wave][j][lane] = s[j];
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * WD_MT + lane - pb.mo;
    if (wave >= nt || i < 0 || i >= pb.M) return;
    double v = sums[0][wave][lane];
#pragma unroll
    for (int q = 1; q < 16; ++q) v += sums[q][wave][lane];
    T *c = nullptr;
    int64_t rs = 0;
#pragma unroll
    for (int j = 0; j < WIDE_TAIL; ++j)
        if (j == wave) {
            c = pb.tc.out[j];
            rs = pb.tc.ors[j];
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

// The operator's chunks of 64 rows x 32 k ahead of the products that read them:
// chunk c of row tile mb at out[(mb * nch + c) * 2048], row r's k .. k + 3 at
// 32 r + k.  Entries before their scale (exact in FP32).  One workgroup per
// chunk, one counter per thread; counters along the rows turn in LDS.
template <bool GAUSS, bool ROWS>
__global__ __launch_bounds__(WD_THR) void wide_pre_kernel(GenMap g, int64_t nch, float *out) {
    __shared__ float t[WD_MT][WD_KC + 1];
    const int tid = threadIdx.x;
    const int64_t mb = blockIdx.x / nch, c = blockIdx.x - mb * nch, m0 = mb * WD_MT, k0 = c * WD_KC;
    const int frow = ROWS ? 4 * (tid & 15) : tid >> 3, fcell = ROWS ? tid >> 4 : tid & 7;
    const uint64_t off = ROWS ? (uint64_t)((g.a_off + k0 + fcell) * g.P + ((g.b_off + m0) >> 2) + (tid & 15))
                              : (uint64_t)((g.a_off + m0 + frow) * g.P + ((g.b_off + k0) >> 2) + fcell);
    float4 v = gen4(GAUSS, ctr_add(g.ctr, off), g.k0, g.k1);
    if constexpr (ROWS) {
#pragma unroll
        for (int e = 0; e < 4; ++e) t[frow + e][fcell] = f4_get(v, e);
        __syncthreads();
        const float *q = &t[tid >> 3][4 * (tid & 7)];
        v = make_float4(q[0], q[1], q[2], q[3]);
    }
    ((float4 *)out)[(int64_t)blockIdx.x * WD_THR + tid] = v;
}

// Scratch, or nullptr when the device cannot provide it, or only by growing it
// while the stream is captured.
static void *try_scratch(int slot, size_t bytes, hipStream_t stream) {
    if (!scratch_usable(slot, bytes, stream)) return nullptr;
    try {
        return scratch(slot, bytes, stream);
    } catch (const Fail &f) {
        if (f.st != RBX_OUT_OF_MEMORY) throw;
        clear_error();
        return nullptr;
    }
}

// Tile width, tail columns, how the tiles and their chunks are shared out, and
// whether the operator is generated ahead.  The time of a workgroup's 32-deep
// chunk is its MFMAs (64 x tile x 32 at the matrix rate, also for columns that do
// not exist) plus the operator's generation (2048 entries, the same for every
// tile width) or the read of one generated ahead, which pays when several
// columns of tiles would generate the same entries.
struct WidePlan {
    int tile, tw;
    bool pre;
    WideWork wk;
    double t;
};
constexpr size_t WIDE_PART_MAX = 16ull << 30;  // bytes of partials: above, tiles are not shared
constexpr size_t WIDE_PRE_MAX = 2ull << 30;    // bytes of an operator generated ahead

template <typename T>
static WidePlan wide_plan(const GemmProblem &pb, int ko, int mo, bool NU, bool split_ok, bool pre_ok) {
    constexpr bool F64 = sizeof(T) == 8;
    // clocks of a CU: 2048 Gaussian entries (measured: 1.2 a clock), chunk overhead,
    // a piece's start and end
    const double gen_here = pb.g.gauss ? 1700.0 : 800.0, gen_pre = 150.0, over = F64 ? 500.0 : 900.0, fixed = 5000.0, mhz = 2100.0;
    const double flop_clk = F64 ? 128.0 : 256.0;
    // FP32 sums have at most 4096 terms, FP64 ones 16384
    const int64_t range_max = (F64 ? 16384 : 4096) / WD_KC;
    const int64_t chunks = (pb.K + ko + WD_KC - 1) / WD_KC;
    const int64_t nMB = (pb.M + mo + WD_MT - 1) / WD_MT;
    RBX_REQUIRE(chunks < (1ll << 31));
    const int64_t cus = num_cus();
    // columns, waves along the rows, blocks per wave (wide_launch_tile)
    static const struct { int cols, wm, cb; } tiles[] = {
        {32, 4, 1},  {64, 2, 1},  {128, 1, 1}, {192, 2, 3}, {256, 1, 2}, {320, 2, 5},
        {384, 1, 3}, {448, 2, 7}, {512, 1, 4}, {640, 1, 5}, {768, 1, 6}, {1024, 1, 8}};
    WidePlan best{};
    best.t = 1e300;
    for (const auto &tl : tiles) {
        const int tile = tl.cols;
        if (F64 && tile > 512) break;
        // (FP32, unit stride along N) the 1024-wide form has too few registers
        if (NU && tile == 1024) break;
        if (NU && pb.N < tl.cb) continue;
        // two waves read the same columns: only where one tile is the whole
        // output (100000 columns, K = 2000, FP32: 448 wide 630 us, 512 wide 590)
        if (tl.wm == 2 && tile > 64 && pb.N > tile) continue;
        const bool two = wide_waves<T>(NU, tl.wm, tl.cb, 0) >= 4;  // two workgroups per CU
        for (int tail = 0; tail < 2; ++tail) {
            int tw = 0;
            if (tail) {
                tw = (int)std::min<int64_t>(pb.N - tile, WIDE_TAIL + 1);
                if (NU || !split_ok || (tile != 128 && tile != 256) || tw < 1 || tw > WIDE_TAIL) continue;
            }
            const int64_t nNB = tail ? 1 : (pb.N + tile - 1) / tile;
            const int64_t tot = nMB * nNB;
            if (tot >= (1ll << 31)) continue;
            for (int pre = 0; pre <= (pre_ok && nNB > 1 ? 1 : 0); ++pre) {
                const double gen = pre ? gen_pre : gen_here;
                const double t_pre = pre ? 6.0 + (double)(nMB * chunks) * 2048.0 / (pb.g.gauss ? 6.5e5 : 1.1e6) : 0.0;
                const double chunk_clk = 64.0 * tile * 64.0 / flop_clk + gen + over + (tw > 1 ? 400.0 : 100.0 * tw);
                // `whole` tiles to one workgroup each, the others to `each`
                auto consider = [&](int64_t whole, int64_t each) {
                    WidePlan p{};
                    WideWork &k = p.wk;
                    const int64_t rest = tot - whole, pieces = rest * each;
                    if (whole + pieces >= (1ll << 31)) return;
                    k.whole = (int)whole;
                    k.rest = (int)rest;
                    k.each = (int)each;
                    k.nMB = (int)nMB;
                    k.chunks = (int)chunks;
                    if (rest > 0) {
                        k.q = (int)(chunks / each);
                        k.r = (int)(chunks % each);
                    }
                    // with two workgroups on a CU the last round overlaps the one before
                    auto rounds = [&](int64_t wgs) {
                        const double up = (double)((wgs + cus - 1) / cus);
                        return two && up > 1 ? std::min(up, (double)wgs / cus + 0.5) : up;
                    };
                    p.t = (whole > 0 ? rounds(whole) * (chunks * chunk_clk + fixed) : 0.0) / mhz + t_pre;
                    if (rest > 0) {
                        const double part = (double)pieces * WD_MT * tile * sizeof(T);
                        if (part > (double)WIDE_PART_MAX) return;
                        p.t += rounds(pieces) * ((double)((chunks + each - 1) / each) * chunk_clk + fixed) / mhz;
                        p.t += 4.0 + part / 3e6;
                    }
                    if (tail) p.t += 3.0;
                    if (p.t >= best.t) return;
                    p.tile = tile;
                    p.tw = tw;
                    p.pre = pre != 0;
                    best = p;
                };
                if (!split_ok || chunks <= range_max) consider(tot, 0);
                if (!split_ok) continue;
                for (int r = 0; r <= 8; ++r) {  // every tile shared
                    int64_t each = std::max((chunks + range_max - 1) / range_max, r * cus / tot);
                    each = std::min(each, chunks);
                    if (each > 1) consider(0, each);
                }
                // whole tiles for as long as every CU has one, the others shared
                const int64_t left = tot % cus;
                if (chunks <= range_max && tot > cus && left > 0)
                    for (int r = 1; r <= 2; ++r) {
                        const int64_t each = std::min(r * cus / left, chunks);
                        if (each > 1) consider(tot - left, each);
                    }
            }
        }
    }
    // partials too large for any number of shares: whole tiles, longer sums
    if (best.tile == 0 && split_ok) return wide_plan<T>(pb, ko, mo, NU, false, pre_ok);
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
    const int64_t nMB = (pb.M + w.mo + WD_MT - 1) / WD_MT;
    const int64_t npre = (w.K + w.ko + WD_KC - 1) / WD_KC;
    const size_t pre_bytes = ((size_t)safe_mul(nMB, npre) + 1) * (WD_MT * WD_KC * sizeof(float));
    // (a materialised operator is read in the same shares as a generated one, so
    // the two give the same bits)
    bool pre_ok = pb.K >= 4 && pre_bytes <= WIDE_PRE_MAX;
    WidePlan p = wide_plan<T>(sized, w.ko, w.mo, NU, true, pre_ok);
    float *pre = nullptr;
    if (p.pre && w.S == nullptr) {
        pre = (float *)try_scratch(SCRATCH_BF16, pre_bytes, stream);
        if (pre == nullptr) p = wide_plan<T>(sized, w.ko, w.mo, NU, true, pre_ok = false);
    }
    char *ws = nullptr;
    size_t part_bytes = 0;
    if (p.wk.rest > 0 || p.tw > 0) {
        const size_t slots = (size_t)p.wk.rest * p.wk.each;
        part_bytes = (slots * WD_MT * p.tile * sizeof(T) + 255) / 256 * 256;
        const size_t tails = slots + (size_t)p.wk.whole;
        ws = (char *)try_scratch(SCRATCH_SPLITK, part_bytes + tails * p.tw * WD_MT * sizeof(T), stream);
        if (ws == nullptr) p = wide_plan<T>(sized, w.ko, w.mo, NU, false, pre_ok && (pre != nullptr || w.S != nullptr));
    }
    RBX_REQUIRE(p.tile > 0);
    w.wk = p.wk;
    w.N = pb.N - p.tw;
    w.part = (T *)ws;
    w.part_cols = w.crs != 1;
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
    if (p.pre && w.S == nullptr) {
        ProfScope prof("wide_pre_kernel", stream);
        const dim3 grid((unsigned)(nMB * npre));  // (below 2^31: WIDE_PRE_MAX)
        if (gauss && rows) hipLaunchKernelGGL((wide_pre_kernel<true, true>), grid, dim3(WD_THR), 0, stream, w.g, npre, pre);
        else if (gauss) hipLaunchKernelGGL((wide_pre_kernel<true, false>), grid, dim3(WD_THR), 0, stream, w.g, npre, pre);
        else if (rows) hipLaunchKernelGGL((wide_pre_kernel<false, true>), grid, dim3(WD_THR), 0, stream, w.g, npre, pre);
        else hipLaunchKernelGGL((wide_pre_kernel<false, false>), grid, dim3(WD_THR), 0, stream, w.g, npre, pre);
        RBX_HIP(hipGetLastError());
        w.pre = pre;
        w.scale = entry_scale<T>(gauss);
    }
    {
        ProfScope prof(sizeof(T) == 8 ? "f64_wide_kernel" : "f32_wide_kernel", stream);
        if (w.S != nullptr && w.srs == 1) wide_launch<T, WIDE_MEM, true>(NU, p.tile, p.tw, w, stream);
        else if (w.S != nullptr) wide_launch<T, WIDE_MEM, false>(NU, p.tile, p.tw, w, stream);
        else if (p.pre) wide_launch<T, WIDE_PRE, false>(NU, p.tile, p.tw, w, stream);
        else if (gauss && rows) wide_launch<T, WIDE_GAUSS, true>(NU, p.tile, p.tw, w, stream);
        else if (gauss) wide_launch<T, WIDE_GAUSS, false>(NU, p.tile, p.tw, w, stream);
        else if (rows) wide_launch<T, WIDE_UNIFORM, true>(NU, p.tile, p.tw, w, stream);
        else wide_launch<T, WIDE_UNIFORM, false>(NU, p.tile, p.tw, w, stream);
        RBX_HIP(hipGetLastError());
    }
    if (p.wk.rest > 0) {
        ProfScope prof(sizeof(T) == 8 ? "f64_reduce_kernel" : "f32_reduce_kernel", stream);
        auto go = [&](auto nw) {
            constexpr int NW = decltype(nw)::value, per = NW < 4 ? 4 : 1;  // sub-blocks of 256 per workgroup
            const int64_t nsub = (WD_MT * p.tile / 256 + per - 1) / per;
            RBX_REQUIRE(p.wk.rest < (1ll << 31) / nsub);
            hipLaunchKernelGGL((wide_reduce_kernel<T, NW>), dim3((unsigned)(p.wk.rest * nsub)),
                               dim3(NW < 4 ? 256 : 64 * NW), 0, stream, w, p.tile, (int)nsub, pb.alpha, pb.beta);
        };
        // enough threads for about 16 waves per CU, at most one per 4 pieces
        const int64_t quads = (int64_t)p.wk.rest * WD_MT * p.tile / 4, want = 256 * 1024;
        const int pieces = p.wk.each;
        if (quads >= want || pieces < 8) go(std::integral_constant<int, 1>{});
        else if (quads * 4 >= want || pieces < 32) go(std::integral_constant<int, 4>{});
        else go(std::integral_constant<int, 16>{});
        RBX_HIP(hipGetLastError());
    }
    if (p.tw > 0) {
        hipLaunchKernelGGL(wide_tail_reduce_kernel<T>, dim3((unsigned)nMB), dim3(1024), 0, stream, w, pb.alpha, pb.beta);
        RBX_HIP(hipGetLastError());
    }
}
template void wide_run<float>(const GemmProblem &, hipStream_t);
template void wide_run<double>(const GemmProblem &, hipStream_t);

}  // namespace rbx
