// U12 of the blocked LU: inverses of a block's 64 x 64 diagonal triangles
// (k_block_linv) and X <- L11^-1 X over a whole outer block (k_u12_block).
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

// L11^-1 of the block's 64 x 64 diagonal triangles (one workgroup each), for
// U12, from the factored block (Lblk, nbo columns): 64 x 64 at
// linv + b * 64 * 64, zero outside the nb x nb triangle.
// By doubling: the four 16 x 16 diagonal inverses, one per wave by
// substitution, then [X11 0; -X22 L21 X11, X22] for the two 32 x 32 blocks
// and for the whole, on MFMA.  It sits on the LU's critical path between a
// block and the next one's update.  One lane per column of the whole
// triangle, 2016 unrolled FMAs, took 35 us, most of it waiting for
// instructions (code that runs once per launch); this takes 6.
template <typename T>
__global__ __launch_bounds__(256)
void k_block_linv(const T *Lblk, int64_t lda, int nbo, T *linv)
{
    typedef typename Mfma16<T>::acc_t acc_t;
    constexpr int LS = NB_IN + 4;
    __shared__ T L[NB_IN][LS], X[NB_IN][LS], W[32][LS];
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lhi = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = min(NB_IN, nbo - (int)blockIdx.x * NB_IN);
    const T *src = Lblk + (int64_t)blockIdx.x * NB_IN * (lda + 1);
    T v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k)
        v[k] = src[(int64_t)min(wave + 4 * k, nb - 1) * lda + min(lane, nb - 1)];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int i = wave + 4 * k;
        L[i][lane] = (i < nb && lane < i) ? v[k] : T(0);
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
            x[i] = s;
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
    T *out = linv + (size_t)blockIdx.x * NB_IN * NB_IN;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int i = wave + 4 * k;
        out[i * NB_IN + lane] = (i < nb && lane < nb) ? X[i][lane] : T(0);
    }
}

// U12 for an outer block of nbo <= NB_OUT rows in one pass.  Each workgroup
// keeps sixteen columns of A12 in LDS and runs the block forward substitution
// on MFMA, sixteen rows of a 64-row panel per wave: for each panel b,
// Y = X_b - sum_{k<b} L_bk X_k, then X_b = Linv_b Y (the panel's inverse,
// from k_block_linv or the panel kernel), with L_bk read from the factored
// block (Lblk = A + K0 * lda + K0).  The operands of L are loaded from memory
// in fragment layout (a lane takes four consecutive k of every sixteen) one
// 64 x 64 stage ahead, and none depends on X.
// Bound by the chain of ten stages and their latency: it precedes the next
// block's update on the LU's critical path.  256 columns take 16 us in FP64
// (47 with the products on FMAs from LDS) and 13 in FP32 (36).
template <typename T>
__global__ __launch_bounds__(256)
void k_u12_block(const T *__restrict__ Lblk, int64_t lda, const T *__restrict__ linv, int nbo,
                 T *B, int64_t ldb, int ncols)
{
    typedef typename Mfma16<T>::acc_t acc_t;
    constexpr int CW = 16, XS = CW + 4;         // four lane groups in different banks
    __shared__ T X[NB_OUT][XS], Y[NB_IN][XS];
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lhi = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c0 = blockIdx.x * CW, nb = (nbo + 63) / 64;
    // stage (b, k): k < b is L_bk, k == b the inverse of panel b
    T cur[16], nxt[16];
    auto load = [&](T (&a)[16], int b, int k) __attribute__((always_inline)) {
        const int row = min(16 * wave + l16, nbo - 64 * b - 1);
        const T *src = (k < b ? Lblk + (int64_t)(64 * b + row) * lda + 64 * k
                              : linv + (size_t)b * NB_IN * NB_IN + row * NB_IN) + 4 * lhi;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) a[4 * q + e] = src[16 * q + e];
    };
    load(cur, 0, 0);
    {
        const int col = min(c0 + (tid & 15), ncols - 1);
        T v[16];
#pragma unroll
        for (int i = 0; i < 16; ++i)
            v[i] = B[(int64_t)min((tid >> 4) + 16 * i, nbo - 1) * ldb + col];
#pragma unroll
        for (int i = 0; i < 16; ++i) X[(tid >> 4) + 16 * i][tid & 15] = v[i];
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
    for (int b = 0; b < nb; ++b) {
        acc_t acc = {0, 0, 0, 0};
        for (int k = 0; k < b; ++k) {
            load(nxt, b, k + 1);
            acc = mul(X + 64 * k, acc);
#pragma unroll
            for (int i = 0; i < 16; ++i) cur[i] = nxt[i];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * wave + Mfma16<T>::drow(lhi, r);
            Y[i][l16] = X[64 * b + i][l16] - acc[r];
        }
        __syncthreads();
        if (b + 1 < nb) load(nxt, b + 1, 0);
        acc = mul(Y, acc_t{0, 0, 0, 0});
#pragma unroll
        for (int i = 0; i < 16; ++i) cur[i] = nxt[i];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 64 * b + 16 * wave + Mfma16<T>::drow(lhi, r);
            X[i][l16] = acc[r];
            if (i < nbo && c0 + l16 < ncols) B[(int64_t)i * ldb + c0 + l16] = acc[r];
        }
        __syncthreads();
    }
}

template <typename T>
int launch_block_linv(la_ctx *ctx, const T *Lblk, int64_t lda, int nbo, T *linv)
{
    hipLaunchKernelGGL(k_block_linv<T>, dim3((unsigned)ceil_div(nbo, NB_IN)), dim3(256), 0,
                       ctx->stream, Lblk, lda, nbo, linv);
    LA_HIP_CHECK(ctx, hipGetLastError());
    return LA_OK;
}

template <typename T>
int launch_u12_block(la_ctx *ctx, const T *Lblk, int64_t lda, const T *linv, int nbo, T *B,
                     int64_t ldb, int64_t ncols)
{
    ProfScope ps(ctx, LA_K_TRSM, (double)nbo * nbo * ncols,
                 (double)sizeof(T) * (2.0 * nbo * ncols + (double)nbo * nbo));
    hipLaunchKernelGGL(k_u12_block<T>, dim3((unsigned)ceil_div(ncols, 16)), dim3(256), 0,
                       ctx->stream, Lblk, lda, linv, nbo, B, ldb, (int)ncols);
    LA_HIP_CHECK(ctx, hipGetLastError());
    return LA_OK;
}

template int launch_block_linv<double>(la_ctx *, const double *, int64_t, int, double *);
template int launch_block_linv<float>(la_ctx *, const float *, int64_t, int, float *);
template int launch_u12_block<double>(la_ctx *, const double *, int64_t, const double *, int,
                                      double *, int64_t, int64_t);
template int launch_u12_block<float>(la_ctx *, const float *, int64_t, const float *, int, float *,
                                     int64_t, int64_t);

}  // namespace lahip
