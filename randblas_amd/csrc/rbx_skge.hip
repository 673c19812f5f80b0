// rbx_skge.hip -- dense sketches lskge3 / rskge3 (skge.hh:154-355) and their
// adjoints, in FP64 and FP32, on the gfx950 matrix cores.
//
// Every call is reduced to one column-major product
//     C[M x N] = alpha * X[M x K] * Y[K x N] + beta * C
// in which exactly one of X, Y is the sketching operator G and the other is
// the dense data D, both addressed through (row stride, column stride).  A
// row-major call is the transposed column-major problem.  When the operator
// is not materialised (buff == NULL) each K-slice of G is generated from its
// Philox counters straight into LDS; G never reaches HBM.
// The product kernels are in rbx_wide.hh; this file holds the entry points,
// the checks and the one-column kernel.
#include "rbx_internal.hh"
#include "rbx_gemm_common.hh"

namespace rbx {

// ---------------------------------------------------------------- one column
// C (M x 1) = alpha * X * y + beta * C with X the generated operator: a
// vector sketch.  The wide kernel would run its MFMAs over 31 empty
// columns; here each workgroup takes GV_ROWS rows and a K range of kw (a
// multiple of 4, chosen so the grid holds several workgroups per CU),
// every thread generates whole Philox cells of those rows (exact values, as
// everywhere) and accumulates v * y in FP64, a fixed-order workgroup
// reduction gives the range's partial, and gemv_reduce_kernel sums the ranges
// in order: deterministic, bound by the generator.  BR = 0: K runs along the
// counter's major index b (one cell = 4 consecutive k of one row); BR = 1: the
// rows run along b (one cell = 4 consecutive rows at one k).
constexpr int GV_ROWS = 8;

template <typename T, int BR>
__global__ __launch_bounds__(256) void gemv_gen_kernel(GenMap g, int64_t M, int64_t K, int64_t kw, const T *y,
                                                       int64_t ys, double *part) {
    __shared__ double red[GV_ROWS][256 / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t r0 = (int64_t)blockIdx.x * GV_ROWS, k0 = (int64_t)blockIdx.y * kw;
    int64_t k1 = k0 + kw;
    if (k1 > K) k1 = K;
    const bool gauss = g.gauss != 0;
    double acc[GV_ROWS];
#pragma unroll
    for (int r = 0; r < GV_ROWS; ++r) acc[r] = 0.0;
    if (BR == 0) {
        const int64_t c0 = k0 / 4, c1 = (k1 + 3) / 4;  // cells of this K range (k0 % 4 == 0)
        for (int64_t c = c0 + tid; c < c1; c += 256) {
            const int64_t k = 4 * c;
            T yv[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) yv[t] = k + t < K ? y[(k + t) * ys] : (T)0;
#pragma unroll
            for (int r = 0; r < GV_ROWS; ++r) {
                if (r0 + r >= M) break;
                const float4 v = gen4(gauss, ctr_add(g.ctr, (uint64_t)((g.a_off + r0 + r) * g.P + (g.b_off >> 2) + c)),
                                      g.k0, g.k1);
#pragma unroll
                for (int t = 0; t < 4; ++t) acc[r] += (double)entry_value<T>(f4_get(v, t), gauss) * (double)yv[t];
            }
        }
    } else {
        // b_off % 4 == 0 and r0 % 8 == 0: the block's rows are cells j = 0, 1
        const int64_t cb = (g.b_off + r0) >> 2;
        for (int64_t k = k0 + tid; k < k1; k += 256) {
            const double yv = (double)y[k * ys];
#pragma unroll
            for (int j = 0; j < GV_ROWS / 4; ++j) {
                if (r0 + 4 * j >= M) break;
                const float4 v = gen4(gauss, ctr_add(g.ctr, (uint64_t)((g.a_off + k) * g.P + cb + j)), g.k0, g.k1);
#pragma unroll
                for (int t = 0; t < 4; ++t) acc[4 * j + t] += (double)entry_value<T>(f4_get(v, t), gauss) * yv;
            }
        }
    }
    // fixed-order reduction: butterfly within each wave, then the waves in order
#pragma unroll
    for (int r = 0; r < GV_ROWS; ++r) {
        double v = acc[r];
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
        if (lane == 0) red[r][wave] = v;
    }
    __syncthreads();
    if (tid < GV_ROWS && r0 + tid < M) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < 4; ++w) v += red[tid][w];
        part[(int64_t)blockIdx.y * M + r0 + tid] = v;
    }
}

template <typename T>
__global__ __launch_bounds__(256) void gemv_reduce_kernel(const double *part, int nk, int64_t M, double alpha,
                                                          double beta, T *C, int64_t crs) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < M; i += (int64_t)gridDim.x * blockDim.x) {
        double v = 0.0;
        for (int z = 0; z < nk; ++z) v += part[(int64_t)z * M + i];
        T *c = C + i * crs;
        double out = alpha * v;
        if (beta != 0.0) out += beta * (double)(*c);
        *c = (T)out;
    }
}

// Runs a one-column problem on gemv_gen_kernel; false when it does not apply.
template <typename T>
static bool gemv_run(const GemmProblem &pb, hipStream_t stream) {
    if (pb.N != 1 || !pb.gen_is_x || pb.sbuf != nullptr || (pb.g.b_off & 3) != 0) return false;
    if (pb.K < 1024) return false;
    const int64_t nb = (pb.M + GV_ROWS - 1) / GV_ROWS;
    if (nb >= (1ll << 31)) return false;
    // K ranges: enough for ~16 workgroups per CU, each 1024 to 16384 deep
    const int64_t want = (16 * (int64_t)num_cus() + nb - 1) / nb;
    int64_t kw = (pb.K + want - 1) / want;
    kw = (kw + 1023) / 1024 * 1024;
    if (kw > 16384) kw = 16384;
    const int64_t nk = (pb.K + kw - 1) / kw;
    if (nk > 65535) return false;
    double *part = (double *)scratch(SCRATCH_SPLITK, (size_t)safe_mul(nk, pb.M) * sizeof(double), stream);
    ProfScope prof("gemv_gen_kernel", stream);
    if (pb.g.b_along_rows)
        hipLaunchKernelGGL((gemv_gen_kernel<T, 1>), dim3((unsigned)nb, (unsigned)nk), dim3(256), 0, stream, pb.g, pb.M,
                           pb.K, kw, (const T *)pb.D, pb.drs, part);
    else
        hipLaunchKernelGGL((gemv_gen_kernel<T, 0>), dim3((unsigned)nb, (unsigned)nk), dim3(256), 0, stream, pb.g, pb.M,
                           pb.K, kw, (const T *)pb.D, pb.drs, part);
    int64_t blocks = (pb.M + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(gemv_reduce_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, stream, (const double *)part,
                       (int)nk, pb.M, pb.alpha, pb.beta, (T *)pb.C, pb.crs);
    RBX_HIP(hipGetLastError());
    return true;
}

// The same product described transposed: C^T = Y^T X^T, so a generated
// operator on the Y side becomes the X side (its orientation flag flips).
static GemmProblem transposed_problem(const GemmProblem &pb) {
    GemmProblem t = pb;
    t.M = pb.N;
    t.N = pb.M;
    t.gen_is_x = pb.gen_is_x ? 0 : 1;
    t.g.b_along_rows = pb.g.b_along_rows ? 0 : 1;
    t.drs = pb.dcs;
    t.dcs = pb.drs;
    t.crs = pb.ccs;
    t.ccs = pb.crs;
    if (pb.sbuf) {
        t.srs = pb.scs;
        t.scs = pb.srs;
    }
    return t;
}

// The operator is the left factor of the wide kernels (one column: of the
// vector kernel); right sketches are the transposed problem.
template <typename T>
static void launch_skge(const GemmProblem &pb, hipStream_t stream) {
    const GemmProblem q = pb.gen_is_x ? pb : transposed_problem(pb);
    if (!gemv_run<T>(q, stream)) wide_run<T>(q, stream);
}

// C = beta * C on an M x N strided matrix (util::safe_scal semantics).
template <typename T>
__global__ __launch_bounds__(256) void scale_kernel(T *C, int64_t M, int64_t N, int64_t crs, int64_t ccs, double beta) {
    int64_t total = M * N;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (int64_t)gridDim.x * blockDim.x) {
        int64_t i = (crs == 1) ? idx % M : idx / N;
        int64_t j = (crs == 1) ? idx / M : idx % N;
        T *c = C + i * crs + j * ccs;
        *c = (beta == 0.0) ? (T)0 : (T)beta * (*c);
    }
}

template <typename T>
void scale_output(T *C, int64_t M, int64_t N, int64_t crs, int64_t ccs, double beta, hipStream_t stream) {
    if (M <= 0 || N <= 0 || beta == 1.0) return;
    int64_t blocks = (M * N + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    ProfScope prof("scale_kernel", stream);
    hipLaunchKernelGGL(scale_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, stream, C, M, N, crs, ccs, beta);
    RBX_HIP(hipGetLastError());
}
template void scale_output<float>(float *, int64_t, int64_t, int64_t, int64_t, double, hipStream_t);
template void scale_output<double>(double *, int64_t, int64_t, int64_t, int64_t, double, hipStream_t);

// Validate a left sketch call exactly as lskge3 does (skge.hh:174-193) and
// build the column-major problem.
template <typename T>
GemmProblem plan_left(char layout, char opS, char opA, int64_t d, int64_t n, int64_t m, double alpha,
                      const rbx_dense_skop *S, int64_t ro_s, int64_t co_s, const T *A, int64_t lda,
                      double beta, T *B, int64_t ldb) {
    RBX_REQUIRE(S != nullptr);
    check_layout(layout);
    check_op(opS);
    check_op(opA);
    RBX_REQUIRE(d >= 0 && n >= 0 && m >= 0);
    RBX_REQUIRE(ro_s >= 0 && co_s >= 0);
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
    GemmProblem pb{};
    pb.alpha = alpha;
    pb.beta = beta;
    pb.D = A;
    pb.C = B;
    // op(A)[k,j] strides in the column-major picture
    if (layout == 'C') {
        pb.M = d; pb.N = n; pb.K = m;
        pb.gen_is_x = 1;
        pb.g = gen_map(*S, opS, ro_s, co_s, false);
        pb.drs = opA == 'N' ? 1 : lda;
        pb.dcs = opA == 'N' ? lda : 1;
        pb.crs = 1; pb.ccs = ldb;
    } else {
        pb.M = n; pb.N = d; pb.K = m;
        pb.gen_is_x = 0;
        pb.g = gen_map(*S, opS, ro_s, co_s, true);
        pb.drs = opA == 'N' ? 1 : lda;
        pb.dcs = opA == 'N' ? lda : 1;
        pb.crs = 1; pb.ccs = ldb;
    }
    set_mem_operand(pb, *S, opS, ro_s, co_s, layout == 'R');
    return pb;
}

// rskge3 (skge.hh:326-346)
template <typename T>
GemmProblem plan_right(char layout, char opA, char opS, int64_t m, int64_t d, int64_t n, double alpha,
                       const T *A, int64_t lda, const rbx_dense_skop *S, int64_t ro_s, int64_t co_s,
                       double beta, T *B, int64_t ldb) {
    RBX_REQUIRE(S != nullptr);
    check_layout(layout);
    check_op(opS);
    check_op(opA);
    RBX_REQUIRE(d >= 0 && n >= 0 && m >= 0);
    RBX_REQUIRE(ro_s >= 0 && co_s >= 0);
    DenseGeom geo = dense_geom(S->dist);
    safe_mul(geo.dim_minor, geo.P);
    int64_t rows_S = opS == 'N' ? n : d, cols_S = opS == 'N' ? d : n;
    RBX_REQUIRE(S->dist.n_rows >= rows_S + ro_s);
    RBX_REQUIRE(S->dist.n_cols >= cols_S + co_s);
    int64_t rows_A = opA == 'N' ? m : n, cols_A = opA == 'N' ? n : m;
    if (layout == 'C') {
        RBX_REQUIRE(lda >= rows_A);
        RBX_REQUIRE(ldb >= m);
    } else {
        RBX_REQUIRE(lda >= cols_A);
        RBX_REQUIRE(ldb >= d);
    }
    GemmProblem pb{};
    pb.alpha = alpha;
    pb.beta = beta;
    pb.D = A;
    pb.C = B;
    if (layout == 'C') {
        pb.M = m; pb.N = d; pb.K = n;
        pb.gen_is_x = 0;
        pb.g = gen_map(*S, opS, ro_s, co_s, false);
        pb.drs = opA == 'N' ? 1 : lda;
        pb.dcs = opA == 'N' ? lda : 1;
        pb.crs = 1; pb.ccs = ldb;
    } else {
        pb.M = d; pb.N = m; pb.K = n;
        pb.gen_is_x = 1;
        pb.g = gen_map(*S, opS, ro_s, co_s, true);
        pb.drs = opA == 'N' ? 1 : lda;
        pb.dcs = opA == 'N' ? lda : 1;
        pb.crs = 1; pb.ccs = ldb;
    }
    set_mem_operand(pb, *S, opS, ro_s, co_s, layout == 'R');
    return pb;
}

template GemmProblem plan_left<float>(char, char, char, int64_t, int64_t, int64_t, double, const rbx_dense_skop *,
                                      int64_t, int64_t, const float *, int64_t, double, float *, int64_t);

template <typename T>
static void run_problem(const GemmProblem &pb, hipStream_t stream) {
    if (pb.M == 0 || pb.N == 0) return;
    if (pb.alpha == 0.0 || pb.K == 0) {
        scale_output<T>((T *)pb.C, pb.M, pb.N, pb.crs, pb.ccs, pb.beta, stream);
        return;
    }
    launch_skge<T>(pb, stream);
}

template <typename T>
bool left_sketch_with_column(char opS, int64_t d, int64_t n, int64_t m, const rbx_dense_skop *S, int64_t ro_s,
                             int64_t co_s, const T *A, int64_t lda, const T *a, T *B, int64_t ldb, T *b,
                             hipStream_t stream) {
    if (d == 0 || m < 4 || S == nullptr || S->buff != nullptr) return false;
    GemmProblem pb = plan_left<T>('C', opS, 'N', d, n + 1, m, 1.0, S, ro_s, co_s, A, lda, 0.0, B, ldb);
    pb.xD = a;
    pb.xdrs = 1;
    pb.xC = b;
    pb.xcrs = 1;
    wide_run<T>(pb, stream);
    return true;
}
template bool left_sketch_with_column<float>(char, int64_t, int64_t, int64_t, const rbx_dense_skop *, int64_t,
                                             int64_t, const float *, int64_t, const float *, float *, int64_t,
                                             float *, hipStream_t);
template bool left_sketch_with_column<double>(char, int64_t, int64_t, int64_t, const rbx_dense_skop *, int64_t,
                                              int64_t, const double *, int64_t, const double *, double *, int64_t,
                                              double *, hipStream_t);

}  // namespace rbx

using namespace rbx;

extern "C" {

rbx_status rbx_slskge3(char layout, char opS, char opA, int64_t d, int64_t n, int64_t m, float alpha,
                       const rbx_dense_skop *S, int64_t ro_s, int64_t co_s, const float *A, int64_t lda,
                       float beta, float *B, int64_t ldb, void *stream) {
    RBX_API_BEGIN
    run_problem<float>(plan_left<float>(layout, opS, opA, d, n, m, alpha, S, ro_s, co_s, A, lda, beta, B, ldb),
                       (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_dlskge3(char layout, char opS, char opA, int64_t d, int64_t n, int64_t m, double alpha,
                       const rbx_dense_skop *S, int64_t ro_s, int64_t co_s, const double *A, int64_t lda,
                       double beta, double *B, int64_t ldb, void *stream) {
    RBX_API_BEGIN
    run_problem<double>(plan_left<double>(layout, opS, opA, d, n, m, alpha, S, ro_s, co_s, A, lda, beta, B, ldb),
                        (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_srskge3(char layout, char opA, char opS, int64_t m, int64_t d, int64_t n, float alpha,
                       const float *A, int64_t lda, const rbx_dense_skop *S, int64_t ro_s, int64_t co_s,
                       float beta, float *B, int64_t ldb, void *stream) {
    RBX_API_BEGIN
    run_problem<float>(plan_right<float>(layout, opA, opS, m, d, n, alpha, A, lda, S, ro_s, co_s, beta, B, ldb),
                       (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_drskge3(char layout, char opA, char opS, int64_t m, int64_t d, int64_t n, double alpha,
                       const double *A, int64_t lda, const rbx_dense_skop *S, int64_t ro_s, int64_t co_s,
                       double beta, double *B, int64_t ldb, void *stream) {
    RBX_API_BEGIN
    run_problem<double>(plan_right<double>(layout, opA, opS, m, d, n, alpha, A, lda, S, ro_s, co_s, beta, B, ldb),
                        (hipStream_t)stream);
    RBX_API_END
}

// Adjoint of B = op(S) * A with respect to A: Abar = op(S)^T * Bbar, i.e. the
// same generated operator read with the opposite op.
rbx_status rbx_slskge3_adjoint(char layout, char opS, int64_t d, int64_t n, int64_t m, float alpha,
                               const rbx_dense_skop *S, int64_t ro_s, int64_t co_s, const float *Bbar,
                               int64_t ldbb, float beta, float *Abar, int64_t ldab, void *stream) {
    RBX_API_BEGIN
    check_op(opS);
    char opT = opS == 'N' ? 'T' : 'N';
    run_problem<float>(plan_left<float>(layout, opT, 'N', m, n, d, alpha, S, ro_s, co_s, Bbar, ldbb, beta, Abar, ldab),
                       (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_dlskge3_adjoint(char layout, char opS, int64_t d, int64_t n, int64_t m, double alpha,
                               const rbx_dense_skop *S, int64_t ro_s, int64_t co_s, const double *Bbar,
                               int64_t ldbb, double beta, double *Abar, int64_t ldab, void *stream) {
    RBX_API_BEGIN
    check_op(opS);
    char opT = opS == 'N' ? 'T' : 'N';
    run_problem<double>(plan_left<double>(layout, opT, 'N', m, n, d, alpha, S, ro_s, co_s, Bbar, ldbb, beta, Abar, ldab),
                        (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_srskge3_adjoint(char layout, char opS, int64_t m, int64_t d, int64_t n, float alpha,
                               const float *Bbar, int64_t ldbb, const rbx_dense_skop *S, int64_t ro_s,
                               int64_t co_s, float beta, float *Abar, int64_t ldab, void *stream) {
    RBX_API_BEGIN
    check_op(opS);
    char opT = opS == 'N' ? 'T' : 'N';
    run_problem<float>(plan_right<float>(layout, 'N', opT, m, n, d, alpha, Bbar, ldbb, S, ro_s, co_s, beta, Abar, ldab),
                       (hipStream_t)stream);
    RBX_API_END
}

rbx_status rbx_drskge3_adjoint(char layout, char opS, int64_t m, int64_t d, int64_t n, double alpha,
                               const double *Bbar, int64_t ldbb, const rbx_dense_skop *S, int64_t ro_s,
                               int64_t co_s, double beta, double *Abar, int64_t ldab, void *stream) {
    RBX_API_BEGIN
    check_op(opS);
    char opT = opS == 'N' ? 'T' : 'N';
    run_problem<double>(plan_right<double>(layout, 'N', opT, m, n, d, alpha, Bbar, ldbb, S, ro_s, co_s, beta, Abar, ldab),
                        (hipStream_t)stream);
    RBX_API_END
}

}  // extern "C"
