// Blocked right-looking Cholesky of a single SPD matrix (row-major, lower).
//
// Semantics of CholeskyDecomposition::new (src/decomp/cholesky.rs:56-110):
//   - any exactly asymmetric pair A[k][j] != A[j][k] (NaN included) -> None
//   - a diagonal pivot d <= 0 -> None (a NaN pivot is NOT rejected: d <= 0 is
//     false for NaN, so the factor carries the NaN on, as the reference does)
//   - the result is the full n x n L with the strict upper triangle zeroed.
// Three-level blocking.  Per 64-column panel: the diagonal block is factored
// by one workgroup and the panel below it is solved against L11^T, sixteen
// rows per wave; the rest of its 256-column middle block gets the panel's
// rank-64 update.  Once a middle block is done, the rest of its 1024-column
// outer block gets one rank-256 update, and once an outer block is done the
// trailing lower triangle gets one rank-1024 update.  Every update is the
// FP64 MFMA GEMM with B = panel^T and the tiles above the diagonal skipped;
// wider ranks amortise reading and writing the trailing triangle.
#include "la_common.hpp"

namespace lahip {

constexpr int PB = 64;          // panel: factored and solved by latency-bound kernels
constexpr int PB_MID = 256;     // middle block: rank of the updates inside an outer block
constexpr int PB_OUT = 1024;    // outer block: rank of the trailing update

// status: bit 1 = asymmetric pair seen.  Compares 64 x 64 tile (bi, bj),
// bi > bj or bi == bj, against its mirror through LDS.
__global__ __launch_bounds__(256)
void k_symcheck(int n, const double *A, int64_t lda, int32_t *flag)
{
    __shared__ double t1[64][65];
    __shared__ double t2[64][65];
    // decode lower-triangular tile index
    const int64_t idx = blockIdx.x;
    int bi = (int)((sqrt(8.0 * (double)idx + 1.0) - 1.0) * 0.5);
    while ((int64_t)bi * (bi + 1) / 2 > idx) --bi;
    while ((int64_t)(bi + 1) * (bi + 2) / 2 <= idx) ++bi;
    const int bj = (int)(idx - (int64_t)bi * (bi + 1) / 2);
    const int r0 = bi * 64, c0 = bj * 64;
    // both tiles' 32 loads per thread from clamped (in-bounds) positions,
    // issued together; positions outside the matrix are never compared
    double v1[16], v2[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int e = threadIdx.x + 256 * k, r = e >> 6, c = e & 63;
        v1[k] = A[(int64_t)min(r0 + r, n - 1) * lda + min(c0 + c, n - 1)];
        v2[k] = A[(int64_t)min(c0 + r, n - 1) * lda + min(r0 + c, n - 1)];
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int e = threadIdx.x + 256 * k, r = e >> 6, c = e & 63;
        t1[r][c] = v1[k];
        t2[r][c] = v2[k];
    }
    __syncthreads();
    int bad = 0;
    for (int e = threadIdx.x; e < 64 * 64; e += 256) {
        int r = e >> 6, c = e & 63;
        if (r0 + r < n && c0 + c < n && (r0 + r) > (c0 + c))
            if (t1[r][c] != t2[c][r]) bad = 1;
    }
    if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr((int *)flag, 1);
}

// v of lane `lane` (a wave-uniform index) to every lane of the wavefront
__device__ inline double potf2_bcast(double v, int lane)
{
    const long long bits = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)bits, lane);
    const int hi = __builtin_amdgcn_readlane((int)(bits >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// sqrt(d) and its reciprocal by Goldschmidt's iteration from v_rsq_f64 (h ->
// 1/(2 sqrt d), g -> sqrt d, both refined by e = 1/2 - h g), g finally
// corrected by its residual: eight dependent operations where sqrt() and a
// division are about thirty.  For d well inside the range of a double.
__device__ inline void sqrt_rcp(double d, double &root, double &rcp)
{
    const double y = __builtin_amdgcn_rsq(d);
    double g = d * y, h = 0.5 * y;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const double e = fma(-h, g, 0.5);
        g = fma(g, e, g);
        h = fma(h, e, h);
    }
    root = fma(fma(-g, g, d), h, g);
    rcp = 2.0 * h;
}
// a / d from rcp = 1 / d to about an ulp, corrected by the residual
__device__ inline double div_rcp(double a, double d, double rcp)
{
    const double q = a * rcp;
    return fma(fma(-q, d, a), rcp, q);
}

constexpr int PT = 16;              // MFMA tile
constexpr int PLS = PB + 4;         // LDS row stride: MFMA fragments of four rows in different banks

// One 16-row tile of X L^T = S for the 16 x 16 lower triangle D (LDS, stride
// PLS, reciprocals of its diagonal in rd): rows S[r][0..16) in LDS, lane r %
// 16 solving row r in registers, in place.
//   x_c = (s_c - sum_{k<c} x_k D[c][k]) / D[c][c], k ascending
// A result that is not finite (an Inf, NaN or zero pivot among the inputs,
// where the corrected quotient may differ from a division) sends the tile
// through the same sum with divisions; the code of that case is out of the
// straight line, which runs once per launch and waits for its instructions.
__device__ inline void solve_tile_right_lt(double *S, const double *D, const double *rd)
{
    const int r = threadIdx.x & 15;
    double x[PT];
#pragma unroll
    for (int c = 0; c < PT; ++c) x[c] = S[r * PLS + c];
    bool ok = true;
#pragma unroll
    for (int c = 0; c < PT; ++c) {
        x[c] = div_rcp(x[c], D[c * PLS + c], rd[c]);
        ok = ok && fabs(x[c]) < INFINITY;
#pragma unroll
        for (int j = c + 1; j < PT; ++j) x[j] = fma(-x[c], D[j * PLS + c], x[j]);
    }
    if (__all(ok)) {
        if ((threadIdx.x & 63) < PT)
#pragma unroll
            for (int c = 0; c < PT; ++c) S[r * PLS + c] = x[c];
    } else if ((threadIdx.x & 63) < PT) {
#pragma unroll 1
        for (int c = 0; c < PT; ++c) {
            double s = S[r * PLS + c];
#pragma unroll 1
            for (int k = 0; k < c; ++k) s = fma(-S[r * PLS + k], D[c * PLS + k], s);
            S[r * PLS + c] = s / D[c * PLS + c];
        }
    }
}

// The 16 x 16 diagonal tile D (LDS) by one wave, in place with zeros above the
// diagonal, and the reciprocals of its diagonal to rd.  Lane r % 16 holds row
// r; column values by readlane.  Returns whether a pivot was <= 0.  Pivots
// outside the range of sqrt_rcp, or results that are not finite, send the
// tile through sqrt() and divisions, in the same order of operations.
__device__ inline bool factor_tile(double *D, double *rd)
{
    const int lane = threadIdx.x & 63, r = lane & 15;
    double x[PT], rc = 0.0;
#pragma unroll
    for (int c = 0; c < PT; ++c) x[c] = D[r * PLS + c];
    bool ok = true;
#pragma unroll
    for (int c = 0; c < PT; ++c) {
        const double d = potf2_bcast(x[c], c);
        ok = ok && d > 1e-280 && d < 1e280;
        double root, rcp;
        sqrt_rcp(d, root, rcp);
        x[c] = r == c ? root : div_rcp(x[c], root, rcp);
        ok = ok && fabs(x[c]) < INFINITY;
        if (r == c) rc = rcp;
        // entries right of the diagonal (rows r < j) are scratch
#pragma unroll
        for (int j = c + 1; j < PT; ++j) x[j] = fma(-x[c], potf2_bcast(x[c], j), x[j]);
    }
    if (__all(ok)) {
        if (lane < PT) {
#pragma unroll
            for (int c = 0; c < PT; ++c) D[r * PLS + c] = c <= r ? x[c] : 0.0;
            rd[r] = rc;
        }
        return false;
    }
    bool bad = false;
#pragma unroll 1
    for (int c = 0; c < PT; ++c) {
        double s = D[r * PLS + c];
#pragma unroll 1
        for (int k = 0; k < c; ++k) s = fma(-D[r * PLS + k], D[c * PLS + k], s);
        const double d = __shfl(s, c);
        if (d <= 0.0) bad = true;
        const double root = sqrt(d);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        if (lane < PT) D[r * PLS + c] = r == c ? root : r > c ? s / root : 0.0;
        if (lane == c) rd[c] = 1.0 / root;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    return bad;
}

// C (16 x 16, LDS) -= A B^T over nk sixteens of columns, A and B sixteen rows
// each (LDS); all with stride PLS.  One wave.
__device__ inline void tile_syrk(double *C, const double *A, const double *B, int nk)
{
    const int lane = threadIdx.x & 63, l16 = lane & 15, lhi = lane >> 4;
    d4_t acc = {0.0, 0.0, 0.0, 0.0};
    for (int k = 0; k < nk; ++k)
#pragma unroll
        for (int s = 0; s < 4; ++s)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[l16 * PLS + 16 * k + 4 * s + lhi],
                                                       B[l16 * PLS + 16 * k + 4 * s + lhi], acc,
                                                       0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) C[(lhi + 4 * r) * PLS + l16] -= acc[r];
}

// The kb x kb diagonal block (kb <= 64) by one workgroup, in LDS, sixteen
// columns at a time: wave 0 factors the 16 x 16 diagonal tile (lane r holds
// row r, column values by readlane), the waves solve the tiles below it, one
// each, and update the rest on MFMA, wave 0 the next diagonal tile first.
//   l[r][c] = (a[r][c] - sum_{k<c} l[r][k] l[c][k]) / sqrt(d_c)
// Bound by the chain through the 64 pivots (square root, reciprocal, column,
// next pivot).  A pivot d <= 0 sets bit 2 of the flag (NaN is not rejected and
// propagates, as in the reference).  One wavefront for the whole block, with
// a library square root and a division per column, took 25 us; this takes 17.
__global__ __launch_bounds__(256)
void k_potf2(double *A, int64_t lda, int kb, int32_t *flag)
{
    __shared__ double a[PB * PLS], rd[PB];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    double v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i)
        v[i] = A[(int64_t)min(wave + 4 * i, kb - 1) * lda + min(lane, kb - 1)];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = wave + 4 * i;         // padding: an identity block
        a[r * PLS + lane] = r < kb && lane <= r ? v[i] : r == lane ? 1.0 : 0.0;
    }
    __syncthreads();
    const int nt = (kb + PT - 1) / PT;
    bool bad = false;
    for (int t = 0; t < nt; ++t) {
        double *D = a + t * PT * (PLS + 1);
        if (wave == 0 && factor_tile(D, rd + t * PT)) bad = true;
        __syncthreads();
        const int below = nt - t - 1;
        if (wave < below)
            solve_tile_right_lt(D + (wave + 1) * PT * PLS, D, rd + t * PT);
        __syncthreads();
        // tiles (i, j), below >= i >= j >= 1, dealt in order: (1, 1) to wave 0
        int w = 0;
        for (int j = 1; j <= below; ++j)
            for (int i = j; i <= below; ++i, w = w == 3 ? 1 : w + 1)
                if (wave == w)
                    tile_syrk(D + i * PT * PLS + j * PT, D + i * PT * PLS, D + j * PT * PLS, 1);
        // wave 0 goes on with its own tile; the others' are not read before the
        // next barrier
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = wave + 4 * i;
        if (r < kb && lane < kb) A[(int64_t)r * lda + lane] = lane <= r ? a[r * PLS + lane] : 0.0;
    }
    if (tid == 0 && bad) atomicOr((int *)flag, 2);
}

// Panel solve: rows of B (nrows x kb, row-major) <- B * L11^-T with L11 the
// kb x kb lower factor at Lm.  A workgroup takes 64 rows, a wave sixteen of
// them, independent of the others: per sixteen columns the product with the
// columns solved so far on MFMA, then the 16 x 16 triangle by substitution,
// one row per lane (the divisions by the diagonal from its reciprocals,
// corrected by the residual).
// Bound by the substitution's chain.  One row per lane through all 64
// columns on one wavefront took 22 us; this takes 12.
__global__ __launch_bounds__(256)
void k_trsm_right_lt(const double *Lm, int64_t ldl, int kb, double *B, int64_t ldb, int nrows)
{
    __shared__ double L[PB * PLS], S[PB * PLS], rd[PB];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row0 = blockIdx.x * PB, c = min(lane, kb - 1);
    double l[16], v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        l[i] = Lm[(int64_t)min(wave + 4 * i, kb - 1) * ldl + c];
        v[i] = B[(int64_t)min(row0 + 16 * wave + i, nrows - 1) * ldb + c];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = wave + 4 * i;         // padding: an identity block
        const double x = r < kb && lane <= r ? l[i] : r == lane ? 1.0 : 0.0;
        L[r * PLS + lane] = x;
        if (lane == r) rd[r] = 1.0 / x;
        S[(16 * wave + i) * PLS + lane] = lane < kb ? v[i] : 0.0;
    }
    __syncthreads();
    double *X = S + 16 * wave * PLS;        // this wave's rows
    const int nt = (kb + PT - 1) / PT;
    for (int t = 0; t < nt; ++t) {
        if (t > 0) tile_syrk(X + t * PT, X, L + t * PT * PLS, t);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        solve_tile_right_lt(X + t * PT, L + t * PT * (PLS + 1), rd + t * PT);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
        if (row0 + 16 * wave + i < nrows && lane < kb)
            B[(int64_t)(row0 + 16 * wave + i) * ldb + lane] = X[i * PLS + lane];
}

__global__ void k_zero_upper(int64_t n, double *A, int64_t lda)
{
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n * n) return;
    int64_t r = e / n, c = e - r * n;
    if (c > r) A[r * lda + c] = 0.0;
}

__global__ void k_flag_to_status(const int32_t *flag, int32_t *status)
{
    int f = *flag;
    *status = (f & 1) ? LA_NOT_SYMMETRIC : ((f & 2) ? LA_NOT_SPD : LA_OK);
}

int potrf_blocked(la_ctx *ctx, int64_t n, double *A, int64_t lda, int32_t *d_status)
{
    if (n <= 0) return LA_OK;
    if (n > INT32_MAX / 2) return set_error(ctx, LA_ERR_ARG, "potrf: n too large");
    int32_t *flag = ctx->d_scratch + SCR_CHOL;
    int fst = fill_i32(ctx, flag, 1, 0);
    if (fst) return fst;
    const int64_t nbt = ceil_div(n, 64);
    hipLaunchKernelGGL(k_symcheck, dim3((unsigned)(nbt * (nbt + 1) / 2)), dim3(256), 0,
                       ctx->stream, (int)n, (const double *)A, lda, flag);
    LA_HIP_CHECK(ctx, hipGetLastError());
    // lower-triangular update of the block whose top-left corner (r0, r0)
    // lies on the diagonal: rows r0..n-1, columns r0..c1-1, minus the
    // product of the factored columns k0..k1-1 of those rows with the
    // transpose of their first c1 - r0 rows
    auto syrk = [&](int64_t r0, int64_t c1, int64_t k0, int64_t k1) -> int {
        const int64_t rows = n - r0, cols = c1 - r0;
        if (rows <= 0 || cols <= 0) return LA_OK;
        const double *P = A + r0 * lda + k0;
        return gemm_rm<double>(ctx, rows, cols, k1 - k0, -1.0, P, lda, P, lda, 1.0,
                               A + r0 * lda + r0, lda, true, true);
    };
    for (int64_t K0 = 0; K0 < n; K0 += PB_OUT) {
        const int64_t K1 = std::min<int64_t>(n, K0 + PB_OUT);
        for (int64_t M0 = K0; M0 < K1; M0 += PB_MID) {
            const int64_t M1 = std::min<int64_t>(K1, M0 + PB_MID);
            for (int64_t k = M0; k < M1; k += PB) {
                const int kb = (int)std::min<int64_t>(PB, M1 - k);
                double *Akk = A + k * lda + k;
                hipLaunchKernelGGL(k_potf2, dim3(1), dim3(256), 0, ctx->stream, Akk, lda, kb,
                                   flag);
                const int64_t below = n - k - kb;
                if (below <= 0) continue;
                hipLaunchKernelGGL(k_trsm_right_lt, dim3((unsigned)ceil_div(below, 64)), dim3(256),
                                   0, ctx->stream, (const double *)Akk, lda, kb,
                                   A + (k + kb) * lda + k, lda, (int)below);
                LA_HIP_CHECK(ctx, hipGetLastError());
                int st = syrk(k + kb, M1, k, k + kb);          // rest of the middle block
                if (st) return st;
            }
            int st = syrk(M1, K1, M0, M1);                      // rest of the outer block
            if (st) return st;
        }
        int st = syrk(K1, n, K0, K1);                           // the trailing triangle
        if (st) return st;
    }
    hipLaunchKernelGGL(k_zero_upper, dim3((unsigned)ceil_div(n * n, 256)), dim3(256), 0,
                       ctx->stream, n, A, lda);
    hipLaunchKernelGGL(k_flag_to_status, dim3(1), dim3(1), 0, ctx->stream, flag, d_status);
    LA_HIP_CHECK(ctx, hipGetLastError());
    return LA_OK;
}

}  // namespace lahip
