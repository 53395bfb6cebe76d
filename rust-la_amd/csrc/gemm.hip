// MFMA GEMM for row-major operands on gfx950.
//
// C[M x N] = alpha * A[M x K] * op(B) + beta * C, every matrix row-major with
// its own leading dimension.  op(B) = B (K x N) or, with TRANS_B, the
// transpose of an N x K row-major matrix.  This one kernel serves the
// drop-in `Mul`/`mmul` (src/matrix/mod.rs:957-980, mmatrix.rs:82-98) and the
// trailing updates of the blocked LU and Cholesky factorisations.
//
// Tiling: 256 threads own a BT x BT tile of C (BT = 128, 64 or 32); their
// four wavefronts each own a quarter of it, in MFMA 16x16 blocks.  K advances
// in slabs of BK staged through double-buffered LDS, k-major (A is transposed
// on the way in), so every MFMA operand fetch is a 16-lane contiguous LDS
// read.  FP64 uses v_mfma_f64_16x16x4f64, FP32 uses v_mfma_f32_16x16x4f32;
// both take A and B as
//   A: lane l holds A[l%16][l/16]        B: lane l holds B[l/16][l%16]
// and return D with lane l, element r holding (measured on gfx950)
//   FP64: D[l/16 + 4*r][l%16]            FP32: D[4*(l/16) + r][l%16].
//
// What bounds it: with many tiles the matrix cores (8192^3: 67 TFLOP/s FP64,
// 132 FP32; 128 x 128 tiles move the least data per operation).  With few,
// the chip is idle: one 128 x 128 FP64 slab of 16 keeps its CU's matrix cores
// busy for 1.7 us, so a 256^3 product on four CUs took 43 us.  So the tile
// shrinks until the tiles fill the CUs, and where even 32 x 32 tiles leave
// one workgroup per CU, KG groups of four wavefronts split K inside the
// workgroup: their slabs overlap each other's load latency, and the partial
// tiles are added pairwise in LDS at the end.  Tile choice in gemm_rm().
#include "la_common.hpp"

namespace lahip {

template <typename T> struct Mfma;
template <> struct Mfma<double> {
    typedef d4_t acc_t;
    // row of accumulator element r held by lane-group lhi = lane/16
    __device__ static inline int drow(int lhi, int r) { return lhi + 4 * r; }
    __device__ static inline acc_t op(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
};
template <> struct Mfma<float> {
    typedef f4_t acc_t;
    __device__ static inline int drow(int lhi, int r) { return 4 * lhi + r; }
    __device__ static inline acc_t op(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
};

// XCD-aware tile order: consecutive workgroup ids are dealt round-robin to
// the 8 XCDs, so remap ids so that each XCD receives a contiguous range of
// logical tiles, then walk tiles in groups of 8 tile-rows for L2 reuse.
__device__ inline void tile_coords(int bid, int ntiles, int tiles_m, int tiles_n,
                                   int &tm, int &tn) {
    int logical = bid;
    if ((ntiles & 7) == 0) {
        int per = ntiles >> 3;
        logical = (bid & 7) * per + (bid >> 3);
    }
    const int G = 8;
    int group = logical / (G * tiles_n);
    int first_m = group * G;
    int gsize = min(tiles_m - first_m, G);
    int in_group = logical - group * G * tiles_n;
    tm = first_m + in_group % gsize;
    tn = in_group / gsize;
}

// Tiles on or below the diagonal (tn <= tm, tn < tiles_n) of a
// lower-triangular update: sum over tm of min(tm + 1, tiles_n).
__host__ __device__ inline int lower_tile_count(int tiles_m, int tiles_n) {
    return tiles_m <= tiles_n ? tiles_m * (tiles_m + 1) / 2
                              : tiles_n * (tiles_n + 1) / 2 + (tiles_m - tiles_n) * tiles_n;
}

// Logical index -> tile of a lower-triangular update, in the order of
// tile_coords restricted to the lower tiles: groups of 8 tile-rows, inside
// a group by column, then by row.  A group holds every row of the columns
// left of its diagonal and a shrinking run of rows for the columns it
// crosses.  The grid enumerates only these tiles, so with the XCD range
// remap every XCD receives an equal, contiguous share of real work.
__device__ inline void lower_tile_coords(int logical, int tiles_m, int tiles_n, int &tm,
                                         int &tn) {
    const int G = 8;
    for (int first_m = 0; first_m < tiles_m; first_m += G) {
        const int gsize = min(G, tiles_m - first_m);
        const int full_cols = min(first_m, tiles_n);
        const int tri = max(0, min(gsize, tiles_n - first_m));
        const int cnt = full_cols * gsize + tri * gsize - tri * (tri - 1) / 2;
        if (logical < cnt) {
            if (logical < full_cols * gsize) {
                tn = logical / gsize;
                tm = first_m + logical % gsize;
                return;
            }
            int o = logical - full_cols * gsize;
            for (int j = 0; j < tri; ++j) {
                const int c = gsize - j;          // rows first_m + j .. first_m + gsize - 1
                if (o < c) {
                    tn = first_m + j;
                    tm = first_m + j + o;
                    return;
                }
                o -= c;
            }
        }
        logical -= cnt;
    }
    tm = tiles_m;
    tn = 0;
}

// BT x BT tile of C per workgroup, K in slabs of BK, KG groups of 256 threads
// that each take a contiguous share of the slabs and add up at the end.
template <typename T, bool TRANS_B, int BT, int BK, int KG>
__global__ __launch_bounds__(256 * KG, KG == 1 ? 2 : 1)
void k_gemm_rm(int M, int N, int K, T alpha, const T *__restrict__ A, int64_t lda,
               const T *__restrict__ B, int64_t ldb, T beta, T *__restrict__ C,
               int64_t ldc, int lower_only, int tiles_m, int tiles_n)
{
    constexpr int PAD = (sizeof(T) == 8) ? 2 : 4;
    constexpr int LD = BT + PAD;
    constexpr int EPT = BT * BK / 256;          // elements per thread, slab and operand
    constexpr int WT = BT / 2, NF = WT / 16;    // wave tile, 16 x 16 blocks along it
    __shared__ __align__(32) T lds[KG][2][2][BK][LD];         // per group: A and B, two slabs each

    int tm, tn;
    if (lower_only) {
        // the grid is the lower tiles rounded up to a multiple of 8
        const int per = gridDim.x >> 3;
        const int logical = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
        if (logical >= lower_tile_count(tiles_m, tiles_n)) return;
        lower_tile_coords(logical, tiles_m, tiles_n, tm, tn);
    } else {
        tile_coords(blockIdx.x, gridDim.x, tiles_m, tiles_n, tm, tn);
    }
    const int m0 = tm * BT, n0 = tn * BT;
    if (tm >= tiles_m || (lower_only && n0 > m0 + BT - 1)) return;

    const int grp = KG == 1 ? 0 : (int)threadIdx.x >> 8;
    const int tid = threadIdx.x & 255;
    T (*const As)[BK][LD] = lds[grp][0], (*const Bs)[BK][LD] = lds[grp][1];
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int l16 = lane & 15, lhi = lane >> 4;

    // global -> register staging assignments, EPT consecutive elements each
    // A tile (BT x BK): thread -> row ar, k offset ak
    constexpr int TPK = BK / EPT, TPN = BT / EPT;
    const int ar = tid / TPK, ak = (tid % TPK) * EPT;
    // B tile: non-trans (BK x BT): row bk_r, columns bc
    //         trans (BT x BK in memory): row (=n) ar, k offset ak
    const int bk_r = tid / TPN, bc = (tid % TPN) * EPT;

    const int nk = (K + BK - 1) / BK;
    const int nkg = (nk + KG - 1) / KG, kt0 = grp * nkg;    // this group's slabs

    T ra[EPT], rb[EPT];
    // Rows of A and columns of B outside the matrices only reach elements of
    // C that are not stored: they are loaded from clamped (in-bounds)
    // positions and left as they are.  Only positions past K are zeroed, in
    // the last slab.  Every load of a tile issues unconditionally.
    const T *const arow = A + (int64_t)min(m0 + ar, M - 1) * lda + ak;
    const T *const btrow = B + (int64_t)min(n0 + ar, N - 1) * ldb + ak;
    const bool full_n = TRANS_B || n0 + BT <= N;
    auto load_tile = [&](int kt) {
        const int k0 = kt * BK;
        if (k0 + BK <= K) {
#pragma unroll
            for (int e = 0; e < EPT; ++e) ra[e] = (arow + k0)[e];
            const T *src = TRANS_B ? btrow + k0 : B + (int64_t)(k0 + bk_r) * ldb + n0 + bc;
            if (full_n) {
#pragma unroll
                for (int e = 0; e < EPT; ++e) rb[e] = src[e];
            } else {
#pragma unroll
                for (int e = 0; e < EPT; ++e) rb[e] = src[min(e, N - 1 - n0 - bc)];
            }
        } else {
            // signed offsets: back from a thread's place into the matrix
#pragma unroll
            for (int e = 0; e < EPT; ++e) ra[e] = arow[min(k0 + e, K - 1 - ak)];
            if (TRANS_B) {
#pragma unroll
                for (int e = 0; e < EPT; ++e) rb[e] = btrow[min(k0 + e, K - 1 - ak)];
            } else {
                const T *src = B + (int64_t)min(k0 + bk_r, K - 1) * ldb + n0 + bc;
#pragma unroll
                for (int e = 0; e < EPT; ++e) rb[e] = src[min(e, N - 1 - n0 - bc)];
            }
#pragma unroll
            for (int e = 0; e < EPT; ++e) {
                if (k0 + ak + e >= K) ra[e] = T(0);
                if (TRANS_B ? k0 + ak + e >= K : k0 + bk_r >= K) rb[e] = T(0);
            }
        }
    };
    auto store_tile = [&](int buf) {
#pragma unroll
        for (int e = 0; e < EPT; ++e) As[buf][ak + e][ar] = ra[e];
        if (!TRANS_B) {
#pragma unroll
            for (int e = 0; e < EPT; ++e) Bs[buf][bk_r][bc + e] = rb[e];
        } else {
#pragma unroll
            for (int e = 0; e < EPT; ++e) Bs[buf][ak + e][ar] = rb[e];
        }
    };

    typedef typename Mfma<T>::acc_t acc_t;
    acc_t acc[NF][NF];
#pragma unroll
    for (int i = 0; i < NF; ++i)
#pragma unroll
        for (int j = 0; j < NF; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = T(0);

    if (nk > 0) {
        load_tile(kt0);
        store_tile(0);
    }
    __syncthreads();
    for (int kt = 0; kt < nkg; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < nkg) load_tile(kt0 + kt + 1);
#pragma unroll
        for (int ks = 0; ks < BK / 4; ++ks) {
            T a[NF], b[NF];
            const int kr = ks * 4 + lhi;
#pragma unroll
            for (int i = 0; i < NF; ++i) a[i] = As[buf][kr][wm * WT + i * 16 + l16];
#pragma unroll
            for (int j = 0; j < NF; ++j) b[j] = Bs[buf][kr][wn * WT + j * 16 + l16];
#pragma unroll
            for (int i = 0; i < NF; ++i)
#pragma unroll
                for (int j = 0; j < NF; ++j) acc[i][j] = Mfma<T>::op(a[i], b[j], acc[i][j]);
        }
        if (kt + 1 < nkg) store_tile(buf ^ 1);
        __syncthreads();
    }
    if constexpr (KG > 1) {
        // sums of the groups, pairwise, through the (now free) slab buffers
        static_assert(sizeof(lds[0]) >= (size_t)BT * BT * sizeof(T), "a group's partial tile");
        acc_t *red = reinterpret_cast<acc_t *>(lds);
        constexpr int GS = BT * BT / 4;
#pragma unroll
        for (int h = KG / 2; h >= 1; h >>= 1) {
            if (grp >= h && grp < 2 * h) {
#pragma unroll
                for (int i = 0; i < NF; ++i)
#pragma unroll
                    for (int j = 0; j < NF; ++j)
                        red[(grp - h) * GS + (i * NF + j) * 256 + tid] = acc[i][j];
            }
            __syncthreads();
            if (grp < h) {
#pragma unroll
                for (int i = 0; i < NF; ++i)
#pragma unroll
                    for (int j = 0; j < NF; ++j)
                        acc[i][j] += red[grp * GS + (i * NF + j) * 256 + tid];
            }
            __syncthreads();
        }
        if (grp > 0) return;
    }

    // epilogue, a block row at a time: C (beta != 0) is read from clamped
    // positions with no per-element condition, so the loads issue together;
    // only stores are guarded (edge tiles, and with lower_only the tiles the
    // diagonal crosses)
    const bool whole = (m0 + BT <= M) && (n0 + BT <= N) && (!lower_only || n0 + BT - 1 <= m0);
#pragma unroll
    for (int i = 0; i < NF; ++i) {
        const int row0 = m0 + wm * WT + i * 16, col0 = n0 + wn * WT + l16;
        T cv[4][NF];
        if (whole) {
            T *cbase = C + (int64_t)row0 * ldc + col0;
            if (beta != T(0)) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int j = 0; j < NF; ++j)
                        cv[r][j] = cbase[(int64_t)Mfma<T>::drow(lhi, r) * ldc + j * 16];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                T *crow = cbase + (int64_t)Mfma<T>::drow(lhi, r) * ldc;
#pragma unroll
                for (int j = 0; j < NF; ++j) {
                    T v = alpha * acc[i][j][r];
                    if (beta != T(0)) v += beta * cv[r][j];
                    crow[j * 16] = v;
                }
            }
            continue;
        }
        if (beta != T(0)) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const T *crow = C + (int64_t)min(row0 + Mfma<T>::drow(lhi, r), M - 1) * ldc;
#pragma unroll
                for (int j = 0; j < NF; ++j) cv[r][j] = crow[min(col0 + j * 16, N - 1)];
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = row0 + Mfma<T>::drow(lhi, r);
            T *crow = C + (int64_t)row * ldc;
#pragma unroll
            for (int j = 0; j < NF; ++j) {
                const int col = col0 + j * 16;
                T v = alpha * acc[i][j][r];
                if (beta != T(0)) v += beta * cv[r][j];
                if (row < M && col < N && (!lower_only || col <= row)) crow[col] = v;
            }
        }
    }
}

template <typename T> struct GemmArgs {
    int M, N, K;
    T alpha;
    const T *A;
    int64_t lda;
    const T *B;
    int64_t ldb;
    T beta;
    T *C;
    int64_t ldc;
    bool lower_only;
};
template <typename T, int BT, int BK, int KG>
static void launch_gemm(hipStream_t s, const GemmArgs<T> &g, bool trans_b)
{
    const int tiles_m = (int)ceil_div(g.M, BT), tiles_n = (int)ceil_div(g.N, BT);
    const int64_t n = g.lower_only ? (int64_t)(lower_tile_count(tiles_m, tiles_n) + 7) / 8 * 8
                                   : (int64_t)tiles_m * tiles_n;
    const dim3 grid((unsigned)n), block(256 * KG);
    if (trans_b)
        hipLaunchKernelGGL((k_gemm_rm<T, true, BT, BK, KG>), grid, block, 0, s, g.M, g.N, g.K,
                           g.alpha, g.A, g.lda, g.B, g.ldb, g.beta, g.C, g.ldc,
                           g.lower_only ? 1 : 0, tiles_m, tiles_n);
    else
        hipLaunchKernelGGL((k_gemm_rm<T, false, BT, BK, KG>), grid, block, 0, s, g.M, g.N, g.K,
                           g.alpha, g.A, g.lda, g.B, g.ldb, g.beta, g.C, g.ldc,
                           g.lower_only ? 1 : 0, tiles_m, tiles_n);
}

template <typename T>
int gemm_rm(la_ctx *ctx, int64_t M, int64_t N, int64_t K, T alpha,
            const T *A, int64_t lda, const T *B, int64_t ldb, T beta,
            T *C, int64_t ldc, bool trans_b, bool lower_only, bool split_k)
{
    if (M <= 0 || N <= 0) return LA_OK;
    if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX)
        return set_error(ctx, LA_ERR_ARG, "gemm: extent exceeds int32");
    if (ceil_div(M, 128) * ceil_div(N, 128) > INT32_MAX / 2)
        return set_error(ctx, LA_ERR_ARG, "gemm: too many tiles");
    const double flop = (lower_only ? 1.0 : 2.0) * (double)M * (double)N * (double)K;
    const double bytes = (double)sizeof(T) * ((double)M * K + (double)K * N +
                                              (beta != T(0) ? 2.0 : 1.0) * (double)M * N);
    ProfScope ps(ctx, sizeof(T) == 8 ? LA_K_GEMM64 : LA_K_GEMM32, flop, bytes);
    const GemmArgs<T> g{(int)M, (int)N, (int)K, alpha, A, lda, B, ldb, beta, C, ldc, lower_only};
    // Tile by the number of tiles against the CUs (P).  Measured, us (FP64,
    // beta = 1, M x N x K; 128 | 64 | 64 K/2 | 64 K/4 | 32 | 32 K/4):
    //   8192^3            16340 | 17008 | 18427 | 20469 | 34210 | 30669
    //   3000 x 3000 x 256   126 |  90.8 |   103 |   132 |   173 |   204
    //   1537 x 777 x 1000   173 |  84.0 |  83.1 |  89.9 |  95.2 |  87.3
    //   1024^3              156 |  55.8 |  52.9 |  47.3 |  76.7 |  70.4
    //   256^3              43.5 |  16.2 |  14.8 |  14.6 |   8.2 |   6.8
    //   64 x 64 x 8192     1323 |   406 |   347 |   312 |   170 |   119
    //   192 x 192 x 64     17.2 |   6.6 |   6.5 |   7.3 |   4.3 |   5.1
    // From four 128-tiles a CU on the large tile's lower traffic wins (FP32
    // 4096 x 4096 x 256: 81 against 87 us for 64); below, 64-tiles do, K
    // split once they leave CUs to one workgroup (under two a CU) and split
    // further when they leave CUs idle and K has slabs to share; and up to
    // two 32-tiles a CU a 64-tile would leave half the chip without work.
    // Every unsplit tile sums an element in the same order (k ascending).
    const int64_t P = ctx->num_cus > 0 ? ctx->num_cus : 256;
    auto tiles = [&](int64_t bt) -> int64_t {
        const int tm = (int)ceil_div(M, bt), tn = (int)ceil_div(N, bt);
        return lower_only && tm < 32768 && tn < 32768 ? lower_tile_count(tm, tn) : (int64_t)tm * tn;
    };
    if (tiles(128) >= 4 * P) {
        launch_gemm<T, 128, 16, 1>(ctx->stream, g, trans_b);
    } else if (tiles(32) <= 2 * P) {
        if (split_k && K >= 192)
            launch_gemm<T, 32, 32, 4>(ctx->stream, g, trans_b);
        else
            launch_gemm<T, 32, 64, 1>(ctx->stream, g, trans_b);
    } else if (!split_k || tiles(64) >= 2 * P) {
        launch_gemm<T, 64, 16, 1>(ctx->stream, g, trans_b);
    } else if (tiles(64) >= P || K < 256) {
        launch_gemm<T, 64, 16, 2>(ctx->stream, g, trans_b);
    } else {
        launch_gemm<T, 64, 16, 4>(ctx->stream, g, trans_b);
    }
    LA_HIP_CHECK(ctx, hipGetLastError());
    return LA_OK;
}

template int gemm_rm<double>(la_ctx *, int64_t, int64_t, int64_t, double, const double *,
                             int64_t, const double *, int64_t, double, double *, int64_t,
                             bool, bool, bool);
template int gemm_rm<float>(la_ctx *, int64_t, int64_t, int64_t, float, const float *,
                            int64_t, const float *, int64_t, float, float *, int64_t, bool,
                            bool, bool);

}  // namespace lahip
