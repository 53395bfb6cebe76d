// Triangular solves with a block of up to 256 rows and many or few columns:
// inverses of its 64 x 64 diagonal triangles (k_block_inv) and X <- T^-1 X
// over the whole block (k_trsm_block).  Used for U12 of the blocked LU, and
// with a GEMM per block for solves with several right-hand sides.
#include "lu_device.hpp"

namespace lahip {

template <typename T> struct Mfma16;
template <> struct Mfma16<double> {
    typedef d4_t acc_t;
    __device__ static inline int drow(int lhi, int r) { return lhi + 4 * r; }
    __device__ static inline acc_t op(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
};
template <> struct Mfma16<float> {
    typedef f4_t acc_t;
    __device__ static inline int drow(int lhi, int r) { return 4 * lhi + r; }
    __device__ static inline acc_t op(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
};

// s / d from rd = 1 / d as a division gives it, the infinite and NaN cases (a
// zero on the diagonal among them) included
template <typename T> __device__ inline T quot(T s, T d, T rd)
{
    const T q = div_rcp(s, d, rd);
    return fabs(q) < T(INFINITY) ? q : s * rd;
}

// Inverses of the 64 x 64 diagonal triangles (one workgroup each) of a packed
// LU whose first nbo columns start at Tm: of L (unit diagonal) or, UPPER, of
// U, which is inverted as its transpose.  64 x 64 at inv + b * 64 * 64, zero
// outside the nb x nb triangle.
// By doubling: the four 16 x 16 diagonal inverses, one per wave by
// substitution, then [X11 0; -X22 L21 X11, X22] for the two 32 x 32 blocks
// and for the whole, on MFMA.  It sits on the LU's critical path between a
// block and the next one's update.  One lane per column of the whole
// triangle, 2016 unrolled FMAs, took 35 us, most of it waiting for
// instructions (code that runs once per launch); this takes 6.
template <typename T, bool UPPER>
__global__ __launch_bounds__(256)
void k_block_inv(const T *Tm, int64_t ldt, int64_t nbo, T *inv)
{
    typedef typename Mfma16<T>::acc_t acc_t;
    constexpr int LS = NB_IN + 4;
    __shared__ T L[NB_IN][LS], X[NB_IN][LS], W[32][LS], dg[NB_IN], rd[NB_IN];
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lhi = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = (int)min((int64_t)NB_IN, nbo - (int64_t)blockIdx.x * NB_IN);
    const T *src = Tm + (int64_t)blockIdx.x * NB_IN * (ldt + 1);
    T v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k)
        v[k] = src[(int64_t)min(wave + 4 * k, nb - 1) * ldt + min(lane, nb - 1)];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int i = wave + 4 * k;
        if (UPPER) {
            L[lane][i] = (lane < nb && i < lane) ? v[k] : T(0);
            if (lane == i) {
                dg[i] = i < nb ? v[k] : T(1);
                rd[i] = i < nb ? T(1) / v[k] : T(1);
            }
        } else {
            L[i][lane] = (i < nb && lane < i) ? v[k] : T(0);
        }
        X[i][lane] = T(0);
    }
    __syncthreads();
    {
        const int d0 = 16 * wave;
        T x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            T s = l16 == i ? T(1) : T(0);
#pragma unroll
            for (int t = 0; t < i; ++t) s -= L[d0 + i][d0 + t] * x[t];
            x[i] = UPPER ? quot(s, dg[d0 + i], rd[d0 + i]) : s;
        }
        if (lane < 16)
#pragma unroll
            for (int i = 0; i < 16; ++i) X[d0 + i][d0 + l16] = x[i];
    }
    __syncthreads();
    // D (16 x 16) = A (rows ra.., columns ca.., K of them) B (rows rb.., columns cb..)
    auto mul = [&](const T (*A)[LS], int ra, int ca, const T (*B)[LS], int rb, int cb,
                   auto k_c) __attribute__((always_inline)) {
        acc_t acc = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < decltype(k_c)::value; k += 4)
            acc = Mfma16<T>::op(A[ra + l16][ca + k + lhi], B[rb + k + lhi][cb + l16], acc);
        return acc;
    };
    if (wave < 2) {
        const int p = 32 * wave;
        const acc_t t = mul(L, p + 16, p, X, p, p, std::integral_constant<int, 16>{});
#pragma unroll
        for (int r = 0; r < 4; ++r) W[16 * wave + Mfma16<T>::drow(lhi, r)][l16] = t[r];
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        const acc_t x = mul(X, p + 16, p + 16, W, 16 * wave, 0, std::integral_constant<int, 16>{});
#pragma unroll
        for (int r = 0; r < 4; ++r) X[p + 16 + Mfma16<T>::drow(lhi, r)][p + l16] = -x[r];
    }
    __syncthreads();
    const int ti = 16 * (wave >> 1), tj = 16 * (wave & 1);
    const acc_t t = mul(L, 32 + ti, 0, X, 0, tj, std::integral_constant<int, 32>{});
#pragma unroll
    for (int r = 0; r < 4; ++r) W[ti + Mfma16<T>::drow(lhi, r)][tj + l16] = t[r];
    __syncthreads();
    const acc_t x = mul(X, 32 + ti, 32, W, 0, tj, std::integral_constant<int, 32>{});
#pragma unroll
    for (int r = 0; r < 4; ++r) X[32 + ti + Mfma16<T>::drow(lhi, r)][tj + l16] = -x[r];
    __syncthreads();
    T *out = inv + (size_t)blockIdx.x * NB_IN * NB_IN;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int i = wave + 4 * k;
        out[i * NB_IN + lane] = (i < nb && lane < nb) ? (UPPER ? X[lane][i] : X[i][lane]) : T(0);
    }
}

// X <- T^-1 X (nbo <= NB_OUT rows, ncols columns at B) for the unit lower or,
// UPPER, the upper triangle of the packed LU block at Tm, in one pass.  Each
// workgroup keeps sixteen columns in LDS and substitutes block by block on
// MFMA, sixteen rows of a 64-row panel per wave: for each panel b in order,
// Y = X_b - sum of T_bk X_k over the panels k done, then X_b = inv(T_bb) Y
// (inv: k_block_inv's or the LU panel kernel's).  The operands of T are
// loaded from memory in fragment layout (a lane takes four consecutive k of
// every sixteen) one 64 x 64 stage ahead, and none depends on X.
// Bound by the chain of ten stages and their latency: as U12 it precedes the
// next block's update on the LU's critical path.  256 columns take 16 us in
// FP64 (47 with the products on FMAs from LDS; 26 with REFINE) and 13 in FP32
// (36).
// REFINE: X_b is corrected once, X_b += inv(T_bb) (Y - T_bb X_b).  The residual
// of a solve with the inverses as they are is 1.0 to 1.3 times that with
// inverses by substitution for random matrices of n <= 512 (2.4 times for
// n = 65 with singular values in [1e-6, 1]); corrected it is below both.
template <typename T, bool UPPER, bool REFINE>
__global__ __launch_bounds__(256)
void k_trsm_block(const T *__restrict__ Tm, int64_t ldt, const T *__restrict__ inv, int nbo,
                  T *B, int64_t ldb, int ncols)
{
    typedef typename Mfma16<T>::acc_t acc_t;
    constexpr int CW = 16, XS = CW + 4;         // four lane groups in different banks
    __shared__ T X[NB_OUT][XS], Y[NB_IN][XS];
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lhi = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c0 = blockIdx.x * CW, nb = (nbo + 63) / 64;
    // panels in order: at(s) is the s-th; stage (s, t): t < s is T_at(s),at(t),
    // t == s the inverse of panel at(s)
    auto at = [&](int s) __attribute__((always_inline)) { return UPPER ? nb - 1 - s : s; };
    T cur[16], nxt[16], ibb[16];
    auto load = [&](T (&a)[16], int s, int t) __attribute__((always_inline)) {
        const int b = at(s), k = at(t), row = min(16 * wave + l16, nbo - 64 * b - 1);
        const T *src = (t < s ? Tm + (int64_t)(64 * b + row) * ldt + 64 * k
                              : inv + (size_t)b * NB_IN * NB_IN + row * NB_IN) + 4 * lhi;
        if (UPPER && t < s && 64 * k + 64 > nbo) {      // the ragged last panel's columns
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int c = 64 * k + 16 * q + 4 * lhi + e;
                    a[4 * q + e] = src[min(16 * q + e, nbo - 1 - 64 * k - 4 * lhi)];
                    if (c >= nbo) a[4 * q + e] = T(0);
                }
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) a[4 * q + e] = src[16 * q + e];
        }
    };
    // T_bb itself, its unit diagonal and the zeros of the other triangle
    auto load_tri = [&](T (&a)[16], int b) __attribute__((always_inline)) {
        const int row = 16 * wave + l16, nbb = min(64, nbo - 64 * b);
        const T *src = Tm + (int64_t)(64 * b + min(row, nbb - 1)) * ldt + 64 * b;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int c = 16 * (k >> 2) + 4 * lhi + (k & 3);
            a[k] = src[min(c, nbb - 1)];
            if (!UPPER && c == row) a[k] = T(1);
            if ((UPPER ? c < row : c > row) || c >= nbb) a[k] = T(0);
        }
    };
    load(cur, 0, 0);
    {
        const int col = min(c0 + (tid & 15), ncols - 1);
        T v[16];
#pragma unroll
        for (int i = 0; i < 16; ++i)
            v[i] = B[(int64_t)min((tid >> 4) + 16 * i, nbo - 1) * ldb + col];
#pragma unroll
        for (int i = 0; i < 16; ++i)
            X[(tid >> 4) + 16 * i][tid & 15] = (tid >> 4) + 16 * i < nbo ? v[i] : T(0);
    }
    __syncthreads();
    auto mul = [&](const T (*x)[XS], acc_t acc) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                acc = Mfma16<T>::op(cur[4 * q + e], x[16 * q + 4 * lhi + e][l16], acc);
        return acc;
    };
    for (int s = 0; s < nb; ++s) {
        const int b = at(s);
        acc_t acc = {0, 0, 0, 0};
        for (int t = 0; t < s; ++t) {
            load(nxt, s, t + 1);
            acc = mul(X + 64 * at(t), acc);
#pragma unroll
            for (int i = 0; i < 16; ++i) cur[i] = nxt[i];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * wave + Mfma16<T>::drow(lhi, r);
            Y[i][l16] = X[64 * b + i][l16] - acc[r];
        }
        __syncthreads();
        if (s + 1 < nb) load(nxt, s + 1, 0);
        acc = mul(Y, acc_t{0, 0, 0, 0});
        if constexpr (REFINE) {
#pragma unroll
            for (int i = 0; i < 16; ++i) ibb[i] = cur[i];
            load_tri(cur, b);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 64 * b + 16 * wave + Mfma16<T>::drow(lhi, r);
                X[i][l16] = i < nbo ? acc[r] : T(0);
            }
            __syncthreads();
            const acc_t tx = mul(X + 64 * b, acc_t{0, 0, 0, 0});
#pragma unroll
            for (int r = 0; r < 4; ++r) Y[16 * wave + Mfma16<T>::drow(lhi, r)][l16] -= tx[r];
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 16; ++i) cur[i] = ibb[i];
            const acc_t d = mul(Y, acc_t{0, 0, 0, 0});
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (fabs(d[r]) < T(INFINITY)) acc[r] += d[r];   // not where X_b overflowed
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) cur[i] = nxt[i];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 64 * b + 16 * wave + Mfma16<T>::drow(lhi, r);
            X[i][l16] = i < nbo ? acc[r] : T(0);
            if (i < nbo && c0 + l16 < ncols) B[(int64_t)i * ldb + c0 + l16] = acc[r];
        }
        __syncthreads();
    }
}

template <typename T>
int launch_block_inv(la_ctx *ctx, bool upper, const T *Tm, int64_t ldt, int64_t n, T *inv)
{
    const dim3 grid((unsigned)ceil_div(n, NB_IN));
    if (upper)
        hipLaunchKernelGGL((k_block_inv<T, true>), grid, dim3(256), 0, ctx->stream, Tm, ldt, n,
                           inv);
    else
        hipLaunchKernelGGL((k_block_inv<T, false>), grid, dim3(256), 0, ctx->stream, Tm, ldt, n,
                           inv);
    LA_HIP_CHECK(ctx, hipGetLastError());
    return LA_OK;
}

template <typename T>
int launch_trsm_block(la_ctx *ctx, bool upper, const T *Tm, int64_t ldt, const T *inv, int nbo,
                      T *B, int64_t ldb, int64_t ncols, bool refine)
{
    ProfScope ps(ctx, LA_K_TRSM, (double)nbo * nbo * ncols,
                 (double)sizeof(T) * (2.0 * nbo * ncols + (double)nbo * nbo));
    const dim3 grid((unsigned)ceil_div(ncols, 16));
    auto k = upper ? (refine ? k_trsm_block<T, true, true> : k_trsm_block<T, true, false>)
                   : (refine ? k_trsm_block<T, false, true> : k_trsm_block<T, false, false>);
    hipLaunchKernelGGL(k, grid, dim3(256), 0, ctx->stream, Tm, ldt, inv, nbo, B, ldb, (int)ncols);
    LA_HIP_CHECK(ctx, hipGetLastError());
    return LA_OK;
}

template int launch_block_inv<double>(la_ctx *, bool, const double *, int64_t, int64_t, double *);
template int launch_block_inv<float>(la_ctx *, bool, const float *, int64_t, int64_t, float *);
template int launch_trsm_block<double>(la_ctx *, bool, const double *, int64_t, const double *,
                                       int, double *, int64_t, int64_t, bool);
template int launch_trsm_block<float>(la_ctx *, bool, const float *, int64_t, const float *, int,
                                      float *, int64_t, int64_t, bool);

}  // namespace lahip
