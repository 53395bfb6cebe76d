// Batched uneven LU with partial pivoting and FP64 iterative refinement in
// one persistent launch.
//
// Problem i: A_i (n_i x n_i, FP64, row-major, n_i <= 1024) and B_i
// (n_i x nrhs_i, nrhs_i <= 8).  One 256-thread workgroup owns a problem from
// start to finish, so no problem ever waits on another workgroup:
//   1. W_i = A_i in the working precision, ||A_i||_inf and max|a| on the way;
//   2. blocked right-looking LU of W_i with partial pivoting: the NB-column
//      panel lives in registers (4 rows per thread, one barrier per column,
//      candidates exchanged through LDS), its row interchanges are applied to
//      the other columns as one permutation of at most 2*NB rows, then
//      U12 = L11^-1 A12 and the update A22 -= L21 U12 on MFMA: of the rest
//      of a 64-column outer block after each panel, of everything to its
//      right once the outer block is done;
//   3. refinement: x = 0, then repeat { r = b - A x in FP64 from A_i;
//      eta = max_c ||r_c|| / (||A|| ||x_c|| + ||b_c||); stop when eta <= tol;
//      solve L U d = P r in working precision (vector in LDS); x += d }.
// Working precisions (template MODE):
//   FP64  W double, NB 16, v_mfma_f64_16x16x4; one solve, eta reported
//   FP32  W float,  NB 32, v_mfma_f32_16x16x4f32
//   FP16  W float,  NB 32, trailing-update operands rounded to FP16: L21 as
//         is (|l| <= 1), U12 after a per-matrix power-of-two scale that puts
//         max|a| in [64, 128) (undone exactly in the epilogue);
//         v_mfma_f32_16x16x32_f16 with FP32 accumulation.
// Each problem is LUDecomposition::new + solve (src/decomp/lu.rs:104-278)
// in structure; pivots follow the reference's rule (largest |v|, lowest row
// on ties) in the working precision.
//
// What bounds it: 4096 problems, n log-uniform in [32, 1024], 1-8 right-hand
// sides, take 23.2 ms in FP32 (FP64 28.9, FP16 36.8; 57, 61.5 and 136 before
// the products with few columns went to MFMA, panels to blocks of eight
// columns and updates to outer blocks of 64).  Of the FP32 time the updates
// are 6.4 ms, panels 4.5, substitution 3.4 and residuals 3.0 (each reads its
// matrix once at about 5 TB/s), conversion 2.0, row moves 2.1, U12 1.5.
#include "lu_device.hpp"
#include <cmath>
#include <utility>

namespace lahip {

constexpr int BL_MAXN = 1024;
constexpr int BL_NT = 256;
constexpr int BL_SLOTS = BL_MAXN / BL_NT;   // panel rows per thread
constexpr int BL_KO = 64;                   // outer block: rank of the trailing update
constexpr int BL_MAXRHS = 8;
constexpr int BL_Y_BYTES = 32768;           // right-hand-side block in LDS
constexpr int BL_STG_BYTES = 36864;         // U12 chunk, x block or diagonal tile
constexpr int BL_BIG = 1 << 30;             // position of an absent row

template <int MODE> struct BlCfg;
template <> struct BlCfg<LA_PREC_FP64> {
    typedef double T; typedef double E;
    static constexpr int NB = 16;
};
template <> struct BlCfg<LA_PREC_FP32> {
    typedef float T; typedef float E;
    static constexpr int NB = 32;
};
template <> struct BlCfg<LA_PREC_FP16> {
    typedef float T; typedef _Float16 E;
    static constexpr int NB = 32;
};

// pivot key: |v| bits + 1, NaN -> 0 (never preferred over a number)
__device__ inline uint64_t bl_key(float v) {
    const uint32_t b = __float_as_uint(v) & 0x7fffffffu;
    return b > 0x7f800000u ? 0ull : (uint64_t)b + 1ull;
}
__device__ inline uint64_t bl_key(double v) {
    const uint64_t b = (uint64_t)__double_as_longlong(v) & 0x7fffffffffffffffull;
    return b > 0x7ff0000000000000ull ? 0ull : b + 1ull;
}
// (key, q) lexicographic with q = ~position: larger |v| first, lower row on ties
__device__ inline bool bl_better(uint64_t k1, uint32_t q1, uint64_t k0, uint32_t q0) {
    return k1 > k0 || (k1 == k0 && q1 > q0);
}
// The wavefront's largest (key, q), to every lane: DPP maxima of the key's
// high word (FP32: of the whole key); lower words and q only among several
// lanes at that maximum.
__device__ inline uint32_t bl_pick_u32(uint32_t v, uint64_t hit) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v,
                                               __ffsll((unsigned long long)hit) - 1);
}
template <typename T> __device__ inline void bl_wave_best(uint64_t &key, uint32_t &q) {
    uint32_t hi = (uint32_t)(key >> 32), lo = (uint32_t)key;
    uint64_t hit;
    if (sizeof(T) == 8) {
        const uint32_t mhi = wave_max_u32(hi);
        hit = __ballot(hi == mhi);
        hi = mhi;
        uint32_t mlo = bl_pick_u32(lo, hit);
        if (__popcll(hit) > 1) {
            mlo = wave_max_u32((hit >> (threadIdx.x & 63)) & 1 ? lo : 0u);
            hit &= __ballot(lo == mlo);
        }
        lo = mlo;
    } else {                        // keys below 2^32
        const uint32_t mlo = wave_max_u32(lo);
        hit = __ballot(lo == mlo);
        lo = mlo;
    }
    uint32_t mq = bl_pick_u32(q, hit);
    if (__popcll(hit) > 1) mq = wave_max_u32((hit >> (threadIdx.x & 63)) & 1 ? q : 0u);
    key = ((uint64_t)hi << 32) | lo;
    q = mq;
}
__device__ inline int bl_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline int64_t bl_uniform(int64_t v) {
    const uint32_t lo = (uint32_t)bl_uniform((int)v), hi = (uint32_t)bl_uniform((int)(v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}
template <typename F, int... I>
__device__ __forceinline__ void bl_for_each(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
__device__ inline float bl_bcast(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ inline double bl_bcast(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// largest of the wave's values, which are not negative and not NaN: their
// bits order as they do
__device__ inline double bl_wave_max(double v) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t hi = (uint32_t)(b >> 32), mhi = wave_max_u32(hi);
    const uint32_t mlo = wave_max_u32(hi == mhi ? (uint32_t)b : 0u);
    return __longlong_as_double((long long)(((uint64_t)mhi << 32) | mlo));
}
__device__ inline double bl_wave_sum(double v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
    return v;
}

__device__ inline double bl_abs_or_inf(double v) { return v == v ? fabs(v) : INFINITY; }

// FP32 / FP64 MFMA, the accumulator row of its element r, and the K batch of
// bl_rows_times
template <typename T> struct BlVec;
template <> struct BlVec<float> {
    typedef f4_t acc_t;
    static constexpr int KB = 128;
    __device__ static inline acc_t mfma(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static inline int drow(int lhi, int r) { return 4 * lhi + r; }
};
template <> struct BlVec<double> {
    typedef d4_t acc_t;
    static constexpr int KB = 64;
    __device__ static inline acc_t mfma(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ static inline int drow(int lhi, int r) { return lhi + 4 * r; }
};

// LDS of one workgroup (about 77 KB: two workgroups fit a CU)
template <int MODE> struct BlLds {
    typedef typename BlCfg<MODE>::T T;
    static constexpr int NB = BlCfg<MODE>::NB;
    __align__(16) unsigned char y[BL_Y_BYTES];       // RHS block, T[n][g], or L11
    __align__(16) unsigned char stg[BL_STG_BYTES];   // U chunk, x block (double[n][g]) or T[64][65]
    T cand_row[2][4][NB];
    uint64_t cand_key[2][4];
    uint32_t cand_q[2][4];
    int mv_src[2 * NB], mv_dst[2 * NB];
    int nmv, prob, singular;
    double red[4 * 2 * BL_MAXRHS];
    double bn[BL_MAXRHS], xn[BL_MAXRHS], rn[BL_MAXRHS];   // max |b_c|, |x_c|, |r_c|
};

// ---------------------------------------------------------------- convert
template <int MODE>
__device__ void bl_convert(int n, const double *__restrict__ Ap,
                           typename BlCfg<MODE>::T *__restrict__ Wp, int *__restrict__ perm,
                           BlLds<MODE> &L, double &anorm, double &amax)
{
    typedef typename BlCfg<MODE>::T T;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double rs_max = 0.0, vmax = 0.0;
    for (int r = wave; r < n; r += 4) {
        double s = 0.0;
        const double *ar = Ap + (int64_t)r * n;
        T *wr = Wp + (int64_t)r * n;
#pragma unroll 4
        for (int c = lane; c < n; c += 64) {
            const double v = ar[c];
            wr[c] = (T)v;
            const double av = fabs(v);
            s += av;
            vmax = fmax(vmax, av);
        }
        rs_max = fmax(rs_max, bl_wave_sum(s));
    }
    for (int i = tid; i < n; i += BL_NT) perm[i] = i;
    vmax = bl_wave_max(vmax);
    // the same values from every lane: a branch here is where the compiler
    // placed spills ahead of the restore of exec
    L.red[wave] = rs_max;
    L.red[4 + wave] = vmax;
    __syncthreads();
    anorm = fmax(fmax(L.red[0], L.red[1]), fmax(L.red[2], L.red[3]));
    amax = fmax(fmax(L.red[4], L.red[5]), fmax(L.red[6], L.red[7]));
    __syncthreads();
}

// ------------------------------------------------------------- factorise
template <int MODE>
__device__ void bl_getrf(int n, typename BlCfg<MODE>::T *__restrict__ W, int *__restrict__ perm,
                         float uscale, BlLds<MODE> &L)
{
    typedef typename BlCfg<MODE>::T T;
    typedef typename BlCfg<MODE>::E E;
    typedef typename BlVec<T>::acc_t acc_t;
    // columns per U12 chunk, its LDS stride, K per MFMA group, column tiles
    // per step.  Strides keep the four lane groups of a fragment read in
    // different LDS banks.
    constexpr int CC = MODE == LA_PREC_FP64 ? 64 : MODE == LA_PREC_FP32 ? 128 : 256;
    constexpr int US = MODE == LA_PREC_FP16 ? BL_KO + 8 : CC + 4;
    constexpr int KS = MODE == LA_PREC_FP16 ? 32 : 16, G = sizeof(T) == 8 ? 4 : 8;
    static_assert((MODE == LA_PREC_FP16 ? CC : BL_KO) * US * sizeof(E) <= BL_STG_BYTES, "U chunk");
    static_assert(BL_KO * BL_KO * sizeof(T) <= BL_Y_BYTES, "L11");
    E *const ustg = reinterpret_cast<E *>(L.stg);
    constexpr int NB = BlCfg<MODE>::NB, NBLK = NB / 8;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lhi = lane >> 4;
    const float uinv = 1.0f / uscale;
    if (tid == 0) L.singular = 0;

    for (int k0 = 0; k0 < n; k0 += NB) {
        const int jb = min(NB, n - k0), m = n - k0;
        const int K0 = k0 / BL_KO * BL_KO, kend = min(n, K0 + BL_KO);   // outer block
        T *Wp = W + (int64_t)k0 * n + k0;
        // ---- panel: rows k0..n-1, columns k0..k0+jb-1, in registers.
        // The column being eliminated is register c of the first block of
        // eight; after eight columns the row arrays rotate left by one block
        // (a finished block moves to the end), so the code is eight columns
        // long, every register index stays static, and only the blocks that
        // still hold active columns are updated.  NB / 8 rotations restore
        // the original column order.  (One column per step with a rotation
        // each and a shuffle tree for the pivot: 10.5 of the 33 ms of 4096
        // FP32 problems, n in [32, 1024]; now 4.5.)
        T a[BL_SLOTS][NB];
        int pos[BL_SLOTS];
#pragma unroll
        for (int s = 0; s < BL_SLOTS; ++s) {
            const int r = tid + BL_NT * s;
            pos[s] = r < m ? r : BL_BIG;
            // unconditional loads from clamped positions, then zeroed
            const T *wr = Wp + (int64_t)min(r, m - 1) * n;
#pragma unroll
            for (int c = 0; c < NB; ++c) a[s][c] = wr[min(c, jb - 1)];
#pragma unroll
            for (int c = 0; c < NB; ++c)
                if (!(r < m && c < jb)) a[s][c] = (T)0;
        }
        if (tid == 0) L.nmv = 0;
        auto column = [&](auto c_c, int it) __attribute__((always_inline)) {
            constexpr int c0 = decltype(c_c)::value;
            const int j = 8 * it + c0;
            if (j >= jb) return;                        // uniform
            const int par = j & 1;
            // largest key of the thread's rows, lowest position on ties
            uint64_t bk = 0;
            uint32_t bq = 0;
#pragma unroll
            for (int s = 0; s < BL_SLOTS; ++s)
                if (pos[s] >= j && pos[s] < m) {
                    const uint64_t kk = bl_key(a[s][c0]);
                    const uint32_t qq = ~(uint32_t)pos[s];
                    if (bl_better(kk, qq, bk, bq)) { bk = kk; bq = qq; }
                }
            bl_wave_best<T>(bk, bq);
            const int wpos = (int)~bq;
#pragma unroll
            for (int s = 0; s < BL_SLOTS; ++s)
                if (pos[s] == wpos && bq != 0) {
#pragma unroll
                    for (int b = 0; b < NBLK; ++b)
                        if (b < NBLK - it) {
#pragma unroll
                            for (int c = 8 * b; c < 8 * b + 8; ++c)
                                L.cand_row[par][wave][c] = a[s][c];
                        }
                }
            if (lane == 0) { L.cand_key[par][wave] = bk; L.cand_q[par][wave] = bq; }
            __syncthreads();
            uint64_t gk = L.cand_key[par][0];
            uint32_t gq = L.cand_q[par][0];
            int gw = 0;
#pragma unroll
            for (int w = 1; w < 4; ++w) {
                const uint64_t k2 = L.cand_key[par][w];
                const uint32_t q2 = L.cand_q[par][w];
                if (bl_better(k2, q2, gk, gq)) { gk = k2; gq = q2; gw = w; }
            }
            const int ppos = (int)~gq;      // current position of the pivot row
            const T *prow = L.cand_row[par][__builtin_amdgcn_readfirstlane(gw)];
            const T piv = prow[c0];
#pragma unroll
            for (int s = 0; s < BL_SLOTS; ++s) {
                if (pos[s] == ppos) pos[s] = j;
                else if (pos[s] == j) pos[s] = ppos;
            }
            if (!(piv != (T)0)) {           // exact zero pivot: no scaling (a NaN scales)
                if (tid == 0) L.singular = 1;
                return;
            }
            const T rinv = (T)1 / piv;
            T l[BL_SLOTS];
#pragma unroll
            for (int s = 0; s < BL_SLOTS; ++s) {
                l[s] = (T)0;
                if (pos[s] > j && pos[s] < m) {
                    l[s] = (MODE == LA_PREC_FP64) ? a[s][c0] / piv : a[s][c0] * rinv;
                    a[s][c0] = l[s];
                }
            }
#pragma unroll
            for (int b = 0; b < NBLK; ++b)
                if (b < NBLK - it) {
                    T u[8];
#pragma unroll
                    for (int c = 0; c < 8; ++c) u[c] = prow[8 * b + c];
#pragma unroll
                    for (int s = 0; s < BL_SLOTS; ++s)
                        if (pos[s] > j && pos[s] < m) {
#pragma unroll
                            for (int c = 0; c < 8; ++c)
                                if (8 * b + c > c0) a[s][8 * b + c] -= l[s] * u[c];
                        }
                }
        };
#pragma unroll 1
        for (int it = 0; it < NBLK; ++it) {
            bl_for_each([&](auto c_c) __attribute__((always_inline)) { column(c_c, it); },
                        std::make_integer_sequence<int, 8>{});
#pragma unroll
            for (int s = 0; s < BL_SLOTS; ++s) {
                T t[8];
#pragma unroll
                for (int c = 0; c < 8; ++c) t[c] = a[s][c];
#pragma unroll
                for (int c = 0; c < NB - 8; ++c) a[s][c] = a[s][c + 8];
#pragma unroll
                for (int c = 0; c < 8; ++c) a[s][NB - 8 + c] = t[c];
            }
        }
        // ---- panel write-back at the final positions, move list
#pragma unroll
        for (int s = 0; s < BL_SLOTS; ++s) {
            const int r = tid + BL_NT * s;
            if (r < m) {
                const int q = pos[s];
                T *dst = Wp + (int64_t)q * n;
#pragma unroll
                for (int c = 0; c < NB; ++c)
                    if (c < jb) dst[c] = a[s][c];
                if (q != r) {
                    const int idx = atomicAdd(&L.nmv, 1);
                    L.mv_src[idx] = r;
                    L.mv_dst[idx] = q;
                }
            }
        }
        __syncthreads();
        const int nmv = __builtin_amdgcn_readfirstlane(L.nmv);
        // ---- the same row permutation on every column outside the panel.
        // A wave owns 64 columns and holds all moved rows of them (at most
        // 2 NB) in registers, so its loads are all in flight together and no
        // barrier parts them from its stores (staged through LDS with two
        // barriers per 64 columns and one load in flight per thread this
        // took 6.4 of the 51 ms of 4096 FP32 problems, n in [32, 1024]; now 2.1).
        if (nmv > 0) {
            const int outside = n - jb;
            for (int x0 = wave * 64; x0 < outside; x0 += BL_NT) {
                const int x = min(x0 + lane, outside - 1), col = x < k0 ? x : x + jb;
                T *const wc = W + (int64_t)k0 * n;       // 32-bit offsets: n <= 1024
                T rv[2 * NB];
#pragma unroll
                for (int e0 = 0; e0 < 2 * NB; e0 += 16)
                    if (e0 < nmv) {
#pragma unroll
                        for (int e = e0; e < e0 + 16; ++e)
                            rv[e] = wc[(uint32_t)(L.mv_src[min(e, nmv - 1)] * n + col)];
                    }
#pragma unroll
                for (int e0 = 0; e0 < 2 * NB; e0 += 16)
                    if (e0 < nmv) {
#pragma unroll
                        for (int e = e0; e < e0 + 16; ++e)
                            if (e < nmv && x0 + lane < outside)
                                wc[(uint32_t)(L.mv_dst[e] * n + col)] = rv[e];
                    }
            }
            int pm = 0;
            if (tid < nmv) pm = perm[k0 + L.mv_src[tid]];
            __syncthreads();
            if (tid < nmv) perm[k0 + L.mv_dst[tid]] = pm;
            __syncthreads();
        }
        // ---- U12 = L11^-1 A12 and A22 -= L21 U12.  After an inner panel: its
        // own rows, on the columns left of the outer block's end.  After the
        // outer block: its BL_KO rows, on every column to the right, so that
        // the trailing matrix is read and written once per BL_KO columns (a
        // pass per NB columns moved 145 GB for 4096 FP64 problems, 26 ms of 60;
        // now 36 GB, 10 ms of 28).
        const bool outer = k0 + jb == kend;
        const int ka = outer ? K0 : k0, kd = k0 + jb - ka;
        const int c_lo = k0 + jb, c_hi = outer ? n : kend;
        if (c_lo >= c_hi) continue;
        // kd is NB or BL_KO here: a shorter panel has no column to its right
        T *l11 = reinterpret_cast<T *>(L.y);                 // [BL_KO][BL_KO]
#pragma unroll
        for (int i0 = 0; i0 < BL_KO; i0 += NB)
            if (i0 < kd) {
                T v[NB / 4];
#pragma unroll
                for (int i = 0; i < NB / 4; ++i)
                    v[i] = W[(uint32_t)((ka + i0 + wave + 4 * i) * n + ka + min(lane, kd - 1))];
#pragma unroll
                for (int i = 0; i < NB / 4; ++i) l11[(i0 + wave + 4 * i) * BL_KO + lane] = v[i];
            }
        __syncthreads();
        for (int u0 = c_lo; u0 < c_hi; u0 += BL_NT) {
            // one column per thread, NB rows at a time: finished rows of the
            // column come back from memory (the thread's own stores)
            const bool valid = u0 + tid < c_hi;
            const int col = min(u0 + tid, c_hi - 1);
            for (int p = 0; p < kd; p += NB) {
                T x[NB];
#pragma unroll
                for (int i = 0; i < NB; ++i) x[i] = W[(uint32_t)((ka + p + i) * n + col)];
                for (int q = 0; q < p; q += NB) {
                    T y[NB];
#pragma unroll
                    for (int k = 0; k < NB; ++k) y[k] = W[(uint32_t)((ka + q + k) * n + col)];
                    const T *lp = l11 + p * BL_KO + q;
#pragma unroll
                    for (int i = 0; i < NB; ++i)
#pragma unroll
                        for (int k = 0; k < NB; ++k) x[i] -= lp[i * BL_KO + k] * y[k];
                }
                const T *lp = l11 + p * BL_KO + p;
#pragma unroll
                for (int i = 1; i < NB; ++i)
#pragma unroll
                    for (int k = 0; k < i; ++k) x[i] -= lp[i * BL_KO + k] * x[k];
                if (valid) {
#pragma unroll
                    for (int i = 0; i < NB; ++i) W[(uint32_t)((ka + p + i) * n + col)] = x[i];
                }
            }
        }
        __syncthreads();
        const int rt_n = (n - c_lo + 15) >> 4;
        for (int cc0 = c_lo; cc0 < c_hi; cc0 += CC) {
            const int cw = min(CC, c_hi - cc0);
            // U chunk to LDS, kd x CC (k-major; FP16: column-major, scaled)
            constexpr int TPR = CC < BL_NT ? CC : BL_NT, RPP = BL_NT / TPR;
            const int uc = tid % TPR, ur = tid / TPR, ucol = cc0 + min(uc, cw - 1);
            for (int k = ur; k < kd; k += 16 * RPP) {
                T v[16];
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    v[i] = W[(uint32_t)((ka + min(k + i * RPP, kd - 1)) * n + ucol)];
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (k + i * RPP < kd) {
                        if constexpr (MODE == LA_PREC_FP16)
                            ustg[uc * US + k + i * RPP] = (E)((float)v[i] * uscale);
                        else
                            ustg[(k + i * RPP) * US + uc] = v[i];
                    }
            }
            __syncthreads();
            // Each wave: one 16-row tile against the chunk's column tiles, G
            // at a time, with the C values of a step loaded together from
            // clamped positions.  Lane group l / 16 takes four (FP16: eight)
            // consecutive k of every sixteen (32), so L21 loads are 16 bytes
            // or more.
            const int ct_n = (cw + 15) >> 4;
            for (int rt = wave; rt < rt_n; rt += 4) {
                const int row0 = c_lo + 16 * rt;
                const T *const lrow = W + (uint32_t)(min(row0 + l16, n - 1) * n + ka);
                h8_t ah[BL_KO / 32];
                T af[BL_KO / 4];
#pragma unroll
                for (int q = 0; q < BL_KO; q += KS)
                    if (q < kd) {
                        T lv[KS / 4];
#pragma unroll
                        for (int e = 0; e < KS / 4; ++e) lv[e] = lrow[q + lhi * (KS / 4) + e];
#pragma unroll
                        for (int e = 0; e < KS / 4; ++e) {
                            if constexpr (MODE == LA_PREC_FP16) ah[q / KS][e] = (_Float16)lv[e];
                            else af[q / 4 + e] = lv[e];
                        }
                    }
                for (int ct0 = 0; ct0 < ct_n; ct0 += G) {
                    T cv[G][4];
                    uint32_t off[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        off[r] = (uint32_t)(min(row0 + BlVec<T>::drow(lhi, r), n - 1) * n);
#pragma unroll
                    for (int g = 0; g < G; ++g) {
                        const int col = min(cc0 + 16 * (ct0 + g) + l16, c_hi - 1);
#pragma unroll
                        for (int r = 0; r < 4; ++r) cv[g][r] = W[off[r] + (uint32_t)col];
                    }
                    // the products of sixteen (32) k are summed, then taken
                    // from C: the sum of all 64 outgrows C and rounds coarser
#pragma unroll
                    for (int q = 0; q < BL_KO; q += KS)
                        if (q < kd) {
                            acc_t acc[G];
#pragma unroll
                            for (int g = 0; g < G; ++g) acc[g] = acc_t{0, 0, 0, 0};
                            if constexpr (MODE == LA_PREC_FP16) {
#pragma unroll
                                for (int g = 0; g < G; ++g)
                                    acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                        ah[q / KS],
                                        *reinterpret_cast<const h8_t *>(
                                            &ustg[(16 * (ct0 + g) + l16) * US + q + 8 * lhi]),
                                        acc[g], 0, 0, 0);
                            } else {
#pragma unroll
                                for (int e = 0; e < 4; ++e)
#pragma unroll
                                    for (int g = 0; g < G; ++g)
                                        acc[g] = BlVec<T>::mfma(
                                            af[q / 4 + e],
                                            ustg[(q + 4 * lhi + e) * US + 16 * (ct0 + g) + l16],
                                            acc[g]);
                            }
#pragma unroll
                            for (int g = 0; g < G; ++g)
#pragma unroll
                                for (int r = 0; r < 4; ++r)
                                    cv[g][r] -= MODE == LA_PREC_FP16 ? (T)(acc[g][r] * uinv) : acc[g][r];
                        }
#pragma unroll
                    for (int g = 0; g < G; ++g) {
                        const int cl = 16 * (ct0 + g) + l16;
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (row0 + BlVec<T>::drow(lhi, r) < n && cl < cw)
                                W[off[r] + (uint32_t)(cc0 + cl)] = cv[g][r];
                    }
                }
            }
            __syncthreads();
        }
    }
}

// ------------------------------------------------ products with few columns
// acc (16 x 16, MFMA layout) += M X over the columns [j0, j1) of 16 rows of M,
// row pointer per lane (row l % 16), X (ldx columns per row, g <= 16 of them)
// in LDS.  Lane group l / 16 takes four consecutive k of every sixteen, so a
// lane loads 16 or 32 consecutive bytes and the rows' cache lines are read
// whole; columns of the result past g are never read.  KB elements of a row
// are loaded while the KB before them are multiplied: these products are
// bound by the way to memory (M is read once), and four rows at a time with
// eight 4- or 8-byte loads in flight reached 1.2 (FP64) and 0.5 TB/s (FP32).
// The sum is short in depth, since it is the residual of the refinement: the
// products of four columns, added pairwise to those of sixteen, which go to
// four accumulators in turn.
template <typename T>
__device__ __forceinline__ typename BlVec<T>::acc_t
bl_rows_times(const T *__restrict__ mrow, const T *X, int ldx, int g, int j0, int j1)
{
    typedef typename BlVec<T>::acc_t acc_t;
    constexpr int KB = BlVec<T>::KB, NC = KB / 16;
    const int lane = threadIdx.x & 63, l16 = lane & 15, lhi = lane >> 4;
    const T *xc = X + min(l16, g - 1);
    acc_t acc[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q] = acc_t{0, 0, 0, 0};
    T v[NC][4], w[NC][4];
    auto load = [&](T (&d)[NC][4], int j) __attribute__((always_inline)) {
        if (j + KB <= j1) {
            const T *src = mrow + j + 4 * lhi;
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) d[c][e] = src[16 * c + e];
        } else {
            // from clamped positions, then zeroed
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) d[c][e] = mrow[min(j + 16 * c + 4 * lhi + e, j1 - 1)];
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (j + 16 * c + 4 * lhi + e >= j1) d[c][e] = T(0);
        }
    };
    if (j0 < j1) load(v, j0);
    for (int j = j0; j < j1; j += KB) {
        if (j + KB < j1) load(w, j + KB);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if (j + 16 * c < j1) {
                acc_t t[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const T x = xc[min(j + 16 * c + 4 * lhi + e, j1 - 1) * ldx];
                    t[e] = BlVec<T>::mfma(v[c][e], x, acc_t{0, 0, 0, 0});
                }
                acc[c & 3] += (t[0] + t[1]) + (t[2] + t[3]);
            }
        }
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[c][e] = w[c][e];
    }
    return (acc[0] + acc[1]) + (acc[2] + acc[3]);
}

// ------------------------------------------------ triangular solves in LDS
// Y (n x g, row-major in LDS) <- L^-1 Y (unit lower), then U^-1 Y, with the
// packed factor in W.  64-row blocks: the off-diagonal part on MFMA, sixteen
// rows per wave; the diagonal tile is loaded (coalesced) before it, staged in
// LDS and solved one row per lane with readlane broadcasts, each wave taking
// right-hand sides c and c + 4 together so that their chains overlap.  The
// chain through the upper tile divides by its diagonal with div_rcp, three
// dependent operations; a result that is not finite is formed again with
// divisions.  (Rows scaled by their reciprocal ahead of the chain would
// leave only the product in it, but u / d leaves the range of T where u x
// and the quotient are ordinary numbers: columns of scales 1e-20 and 1e20.)
template <typename T>
__device__ void bl_trsv_lu(int n, const T *__restrict__ W, T *Y, int g, unsigned char *stg)
{
    T (*D)[65] = reinterpret_cast<T (*)[65]>(stg);
    static_assert(sizeof(T) * 64 * 65 <= BL_STG_BYTES, "diagonal tile");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lhi = lane >> 4;
    const int nblk = (n + 63) / 64;
    for (int step = 0; step < 2 * nblk; ++step) {
        const bool fwd = step < nblk;
        const int b0 = 64 * (fwd ? step : 2 * nblk - 1 - step), bs = min(64, n - b0);
        T dv[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int r = (tid >> 6) + 4 * q;
            dv[q] = W[(int64_t)(b0 + min(r, bs - 1)) * n + b0 + min(lane, bs - 1)];
        }
        const int j0 = fwd ? 0 : b0 + bs, j1 = fwd ? b0 : n;
        if (j0 < j1) {
            const T *mrow = W + (int64_t)(b0 + min(16 * wave + l16, bs - 1)) * n;
            const auto acc = bl_rows_times<T>(mrow, Y, g, g, j0, j1);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 16 * wave + BlVec<T>::drow(lhi, r);
                if (i < bs && l16 < g) Y[(b0 + i) * g + l16] -= acc[r];
            }
        }
#pragma unroll
        for (int q = 0; q < 16; ++q) D[(tid >> 6) + 4 * q][lane] = dv[q];
        __syncthreads();
        if (wave < g) {
            const int i = min(lane, bs - 1);
            const bool two = wave + 4 < g;
            T *y0p = Y + (b0 + i) * g + wave, *y1p = y0p + (two ? 4 : 0);
            T y0 = *y0p, y1 = *y1p;
            T row[64];
#pragma unroll
            for (int k = 0; k < 64; ++k) row[k] = D[i][k];
            if (fwd) {
#pragma unroll
                for (int k = 0; k < 63; ++k)
                    if (k + 1 < bs) {
                        const T a = bl_bcast(y0, k), b = bl_bcast(y1, k);
                        const T l = i > k ? row[k] : (T)0;
                        if (i > k) { y0 -= l * a; y1 -= l * b; }
                    }
            } else {
                const T d = D[i][i], rd = (T)1 / d, s0 = y0, s1 = y1;
#pragma unroll
                for (int k = 63; k >= 0; --k)
                    if (k < bs) {
                        const T q0 = div_rcp(y0, d, rd), q1 = div_rcp(y1, d, rd);
                        if (i == k) { y0 = q0; y1 = q1; }
                        const T a = bl_bcast(y0, k), b = bl_bcast(y1, k);
                        if (i < k) { y0 -= row[k] * a; y1 -= row[k] * b; }
                    }
                if (__any(!(fabs(y0) < (T)INFINITY && fabs(y1) < (T)INFINITY))) {
                    y0 = s0;
                    y1 = s1;
#pragma unroll 1
                    for (int k = bs - 1; k >= 0; --k) {
                        if (i == k) { y0 = y0 / d; y1 = y1 / d; }
                        const T a = bl_bcast(y0, k), b = bl_bcast(y1, k), u = D[i][k];
                        if (i < k) { y0 -= u * a; y1 -= u * b; }
                    }
                }
            }
            if (lane < bs) {
                *y0p = y0;
                if (two) *y1p = y1;
            }
        }
        __syncthreads();
    }
}

// ----------------------------------------------------------- refinement
// r = b - A x (FP64) for the rows in pivot order; Y[i][c] = r[perm[i]][c]
// in working precision; L.rn[c] = max |r_c|, a NaN counted as infinite (fmax
// would drop it, and a NaN residual would pass for none).  Sixteen rows per
// wave at a time on FP64 MFMA.
template <int MODE>
__device__ void bl_residual(int n, int nrhs, int c0, int g, bool first,
                            const double *__restrict__ Ap, const double *__restrict__ Bp,
                            const double *Xp, const int *__restrict__ perm, BlLds<MODE> &L)
{
    typedef typename BlCfg<MODE>::T T;
    T *Y = reinterpret_cast<T *>(L.y);
    double *xs = reinterpret_cast<double *>(L.stg);      // x block, [j][g], in LDS
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lhi = lane >> 4;
    if (!first) {
        for (int e = tid; e < n * g; e += BL_NT) {
            const int j = e / g, c = e - j * g;
            xs[e] = Xp[(int64_t)j * nrhs + c0 + c];
        }
        __syncthreads();
    }
    double rmax = 0.0;                                   // of column l16
    for (int i0 = wave * 16; i0 < n; i0 += 64) {
        // right-hand sides of the rows this lane ends up with
        double bv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            bv[r] = Bp[(int64_t)perm[min(i0 + BlVec<double>::drow(lhi, r), n - 1)] * nrhs + c0 +
                       min(l16, g - 1)];
        d4_t acc = {0.0, 0.0, 0.0, 0.0};
        if (!first)
            acc = bl_rows_times<double>(Ap + (int64_t)perm[min(i0 + l16, n - 1)] * n, xs, g, g, 0,
                                        n);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = i0 + BlVec<double>::drow(lhi, r);
            if (i < n && l16 < g) {
                const double v = bv[r] - acc[r];
                Y[i * g + l16] = (T)v;
                rmax = fmax(rmax, bl_abs_or_inf(v));
            }
        }
    }
    rmax = fmax(rmax, __shfl_xor(rmax, 16));
    rmax = fmax(rmax, __shfl_xor(rmax, 32));
    if (lane < BL_MAXRHS) L.red[wave * BL_MAXRHS + lane] = rmax;
    __syncthreads();
    if (tid < BL_MAXRHS)
        L.rn[tid] = fmax(fmax(L.red[tid], L.red[BL_MAXRHS + tid]),
                         fmax(L.red[2 * BL_MAXRHS + tid], L.red[3 * BL_MAXRHS + tid]));
    __syncthreads();
}

// x += Y (columns c0..c0+g-1); L.xn[c] = max |x_c| afterwards (NaN: infinite)
template <int MODE>
__device__ void bl_update_x(int n, int nrhs, int c0, int g, double *Xp, BlLds<MODE> &L,
                            bool first)
{
    typedef typename BlCfg<MODE>::T T;
    const T *Y = reinterpret_cast<const T *>(L.y);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double xm[BL_MAXRHS];
#pragma unroll
    for (int c = 0; c < BL_MAXRHS; ++c) xm[c] = 0.0;
    for (int e = tid; e < n * g; e += BL_NT) {
        const int i = e / g, c = e - i * g;
        double *xp = Xp + (int64_t)i * nrhs + c0 + c;
        const double v = (first ? 0.0 : *xp) + (double)Y[e];
        *xp = v;
#pragma unroll
        for (int q = 0; q < BL_MAXRHS; ++q)
            if (q == c) xm[q] = fmax(xm[q], bl_abs_or_inf(v));
    }
#pragma unroll
    for (int c = 0; c < BL_MAXRHS; ++c) {
        const double v = bl_wave_max(xm[c]);
        L.red[4 * BL_MAXRHS + wave * BL_MAXRHS + c] = v;
    }
    __syncthreads();
    if (tid < BL_MAXRHS)
        L.xn[tid] = fmax(fmax(L.red[4 * BL_MAXRHS + tid], L.red[5 * BL_MAXRHS + tid]),
                         fmax(L.red[6 * BL_MAXRHS + tid], L.red[7 * BL_MAXRHS + tid]));
    __syncthreads();
}

template <int MODE>
__device__ void bl_refine(int n, int nrhs, const double *__restrict__ Ap,
                          const double *__restrict__ Bp, double *Xp,
                          const typename BlCfg<MODE>::T *__restrict__ W,
                          const int *__restrict__ perm, double anorm, double tol, int max_iter,
                          BlLds<MODE> &L, int &status, int &iters, double &eta_out)
{
    typedef typename BlCfg<MODE>::T T;
    T *Y = reinterpret_cast<T *>(L.y);
    const int cap = BL_Y_BYTES / (int)sizeof(T);
    const int xcap = BL_STG_BYTES / (int)sizeof(double);
    const int gmax = max(1, min(min(nrhs, BL_MAXRHS), min(cap, xcap) / n));
    status = LA_OK;
    iters = 0;
    eta_out = 0.0;
    for (int c0 = 0; c0 < nrhs; c0 += gmax) {
        const int g = min(gmax, nrhs - c0);
        double eta = 1.0, eta_prev = 1e300;
        int stalls = 0, it = 0;
        for (;; ++it) {
            bl_residual<MODE>(n, nrhs, c0, g, it == 0, Ap, Bp, Xp, perm, L);
            if (it == 0) {
                if (threadIdx.x < BL_MAXRHS) {
                    L.bn[threadIdx.x] = L.rn[threadIdx.x];
                    L.xn[threadIdx.x] = 0.0;
                }
                __syncthreads();
            }
            eta = 0.0;
            for (int c = 0; c < g; ++c) {
                const double den = anorm * L.xn[c] + L.bn[c], r = L.rn[c];
                const double e = den > 0.0 ? r / den : (r > 0.0 ? 1e300 : 0.0);
                eta = (e != e) ? 1e300 : fmax(eta, e);
            }
            if (it > 0) {
                if (eta <= tol) break;
                if (MODE == LA_PREC_FP64) break;
                if (it > max_iter) { status = LA_NOT_CONVERGED; break; }
                if (eta > 0.5 * eta_prev) {
                    if (++stalls >= 3) { status = LA_NOT_CONVERGED; break; }
                } else {
                    stalls = 0;
                }
            }
            eta_prev = eta;
            bl_trsv_lu<T>(n, W, Y, g, L.stg);
            bl_update_x<MODE>(n, nrhs, c0, g, Xp, L, it == 0);
        }
        iters = max(iters, it - 1);
        eta_out = fmax(eta_out, eta);
    }
}

// ---------------------------------------------------------------- kernel
template <int MODE>
__global__ __launch_bounds__(BL_NT, 2)
void k_lu_ir_batched(int count, const int32_t *__restrict__ order, const int32_t *__restrict__ nvec,
                     const int32_t *__restrict__ rhsvec, const int64_t *__restrict__ offA,
                     const int64_t *__restrict__ offB, const int64_t *__restrict__ offW,
                     const int64_t *__restrict__ offN, const double *A, const double *B, double *X,
                     typename BlCfg<MODE>::T *Wbuf, int32_t *permbuf, double tol, int max_iter,
                     int32_t *status, int32_t *iters, double *berr, uint32_t *queue)
{
    __shared__ BlLds<MODE> L;
    for (;;) {
        if (threadIdx.x == 0) L.prob = (int)atomicAdd(&queue[0], 1u);
        __syncthreads();
        // Uniform, so that nothing derived from it is spilled early: a spill at
        // the end of a divergent branch was placed ahead of the restore of
        // exec, which keeps the branch's lanes only.  (With the body under an
        // if instead of the continue below, every loop becomes a scalar branch
        // and 4096 FP32 problems take 26.1 ms instead of 23.2.)
        const int pi = __builtin_amdgcn_readfirstlane(L.prob);
        __syncthreads();
        if (pi >= count) break;
        const int prob = bl_uniform(order[pi]);
        const int n = bl_uniform(nvec[prob]), nrhs = bl_uniform(rhsvec[prob]);
        if (n <= 0 || n > BL_MAXN || nrhs <= 0 || nrhs > BL_MAXRHS) {
            if (threadIdx.x == 0) {
                status[prob] = LA_ERR_SHAPE;
                iters[prob] = 0;
                berr[prob] = 0.0;
            }
            continue;
        }
        const double *Ap = A + bl_uniform(offA[prob]);
        const double *Bp = B + bl_uniform(offB[prob]);
        double *Xp = X + bl_uniform(offB[prob]);
        typename BlCfg<MODE>::T *Wp = Wbuf + bl_uniform(offW[prob]);
        int *perm = permbuf + bl_uniform(offN[prob]);
        double anorm, amax;
        bl_convert<MODE>(n, Ap, Wp, perm, L, anorm, amax);
        float uscale = 1.0f;
        if (MODE == LA_PREC_FP16 && amax > 0.0 && amax < 1e300)
            uscale = ldexpf(1.0f, 6 - ilogb(amax));
        bl_getrf<MODE>(n, Wp, perm, uscale, L);
        __syncthreads();
        const int sing = L.singular;
        int st = LA_SINGULAR, it = 0;
        double eta = 0.0;
        if (!sing) bl_refine<MODE>(n, nrhs, Ap, Bp, Xp, Wp, perm, anorm, tol, max_iter, L, st, it, eta);
        if (threadIdx.x == 0) {
            status[prob] = st;
            iters[prob] = it;
            berr[prob] = eta;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const unsigned d = atomicAdd(&queue[1], 1u);
        if (d == gridDim.x - 1) {
            atomicExch(&queue[0], 0u);
            atomicExch(&queue[1], 0u);
        }
    }
}

static const void *lu_ir_kernel(int prec) {
    switch (prec) {
    case LA_PREC_FP64: return (const void *)k_lu_ir_batched<LA_PREC_FP64>;
    case LA_PREC_FP32: return (const void *)k_lu_ir_batched<LA_PREC_FP32>;
    case LA_PREC_FP16: return (const void *)k_lu_ir_batched<LA_PREC_FP16>;
    default: return nullptr;
    }
}

int lu_ir_batched_grid(la_ctx *ctx, int prec)
{
    const void *k = lu_ir_kernel(prec);
    int per_cu = 0;
    if (!k || hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, BL_NT, 0) != hipSuccess ||
        per_cu < 1)
        per_cu = 1;
    (void)hipGetLastError();
    return std::max(1, ctx->num_cus) * per_cu;
}

int launch_lu_ir_batched(la_ctx *ctx, hipStream_t s, int prec, int grid, int count,
                         const int32_t *order, const int32_t *nvec, const int32_t *rhsvec,
                         const int64_t *offA, const int64_t *offB, const int64_t *offW,
                         const int64_t *offN, const double *A, const double *B, double *X,
                         void *Wbuf, int32_t *permbuf, double tol, int max_iter, int32_t *status,
                         int32_t *iters, double *berr, uint32_t *queue)
{
    switch (prec) {
    case LA_PREC_FP64:
        hipLaunchKernelGGL(k_lu_ir_batched<LA_PREC_FP64>, dim3(grid), dim3(BL_NT), 0, s, count,
                           order, nvec, rhsvec, offA, offB, offW, offN, A, B, X, (double *)Wbuf,
                           permbuf, tol, max_iter, status, iters, berr, queue);
        break;
    case LA_PREC_FP32:
        hipLaunchKernelGGL(k_lu_ir_batched<LA_PREC_FP32>, dim3(grid), dim3(BL_NT), 0, s, count,
                           order, nvec, rhsvec, offA, offB, offW, offN, A, B, X, (float *)Wbuf,
                           permbuf, tol, max_iter, status, iters, berr, queue);
        break;
    case LA_PREC_FP16:
        hipLaunchKernelGGL(k_lu_ir_batched<LA_PREC_FP16>, dim3(grid), dim3(BL_NT), 0, s, count,
                           order, nvec, rhsvec, offA, offB, offW, offN, A, B, X, (float *)Wbuf,
                           permbuf, tol, max_iter, status, iters, berr, queue);
        break;
    default:
        return set_error(ctx, LA_ERR_ARG, "batched LU-IR: precision must be FP64, FP32 or FP16");
    }
    LA_HIP_CHECK(ctx, hipGetLastError());
    return LA_OK;
}

// ------------------------------------------------------------- generator
// Batch of A_i = U_i diag(sigma) V_i^T (Householder products, as
// la_gen_svd_matrix_dev) with B_i standard normal (n_i x nrhs_i) and the
// exact solutions X*_i = V_i diag(1/sigma) U_i^T B_i.  Problem p draws its
// reflector vectors from streams stream_base + 256 p + i (U) and
// stream_base + 256 p + 128 + i (V), i < nrefl <= 128, and B_i from stream
// stream_base + 256 p + 255 (row-major order).  One workgroup per problem.
__device__ inline double bl_normal_at(uint64_t key, int64_t e) {
    const int64_t p = e >> 1;
    const double two_pi = 6.283185307179586476925286766559;
    const double u1 = (double)((mix64(key + (uint64_t)(2 * p + 1) * GOLDEN) >> 11) + 1) * 0x1.0p-53;
    const double u2 = (double)(mix64(key + (uint64_t)(2 * p + 2) * GOLDEN) >> 11) * 0x1.0p-53;
    const double r = sqrt(-2.0 * log(u1));
    const double t = two_pi * u2;
    return (e & 1) ? r * sin(t) : r * cos(t);
}

__device__ double bl_load_reflector(uint64_t seed, uint64_t stream, int n, double *v, double *red)
{
    const uint64_t key = mix64(seed + (stream + 1) * GOLDEN);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double s = 0.0;
    for (int i = tid; i < n; i += BL_NT) {
        const double x = bl_normal_at(key, i);
        v[i] = x;
        s += x * x;
    }
    s = bl_wave_sum(s);
    if (lane == 0) red[wave] = s;
    __syncthreads();
    const double vtv = red[0] + red[1] + red[2] + red[3];
    __syncthreads();
    return vtv;
}

__global__ __launch_bounds__(BL_NT)
void k_gen_svd_batch(int count, const int32_t *nvec, const int32_t *rhsvec, const int64_t *offA,
                     const int64_t *offB, double kappa, int nrefl, uint64_t seed,
                     uint64_t stream_base, double *A, double *B, double *Xs)
{
    __shared__ double v[BL_MAXN], w[BL_MAXN], red[8];
    const int prob = blockIdx.x;
    if (prob >= count) return;
    const int n = nvec[prob], nrhs = rhsvec[prob];
    if (n <= 0 || n > BL_MAXN || nrhs <= 0 || nrhs > BL_MAXRHS) return;
    double *Ap = A + offA[prob];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t base = stream_base + 256ull * (uint64_t)prob;
    auto sigma = [&](int i) { return n > 1 ? pow(kappa, -(double)i / (double)(n - 1)) : 1.0; };
    for (int64_t e = tid; e < (int64_t)n * n; e += BL_NT) {
        const int r = (int)(e / n), c = (int)(e - (int64_t)r * n);
        Ap[e] = r == c ? sigma(r) : 0.0;
    }
    __syncthreads();
    for (int i = nrefl - 1; i >= 0; --i) {           // A <- H_i A
        const double vtv = bl_load_reflector(seed, base + i, n, v, red);
        const double f = 2.0 / vtv;
        for (int c = tid; c < n; c += BL_NT) {
            double s = 0.0;
            for (int r = 0; r < n; ++r) s += v[r] * Ap[(int64_t)r * n + c];
            w[c] = s;
        }
        __syncthreads();
        for (int64_t e = tid; e < (int64_t)n * n; e += BL_NT) {
            const int r = (int)(e / n), c = (int)(e - (int64_t)r * n);
            Ap[e] -= f * v[r] * w[c];
        }
        __syncthreads();
    }
    for (int i = nrefl - 1; i >= 0; --i) {           // A <- A H'_i
        const double vtv = bl_load_reflector(seed, base + 128 + i, n, v, red);
        const double f = 2.0 / vtv;
        for (int r = wave; r < n; r += 4) {
            double s = 0.0;
            for (int c = lane; c < n; c += 64) s += Ap[(int64_t)r * n + c] * v[c];
            s = bl_wave_sum(s);
            if (lane == 0) w[r] = s;
        }
        __syncthreads();
        for (int64_t e = tid; e < (int64_t)n * n; e += BL_NT) {
            const int r = (int)(e / n), c = (int)(e - (int64_t)r * n);
            Ap[e] -= f * w[r] * v[c];
        }
        __syncthreads();
    }
    // right-hand sides and exact solutions
    double *Bp = B + offB[prob], *Xp = Xs + offB[prob];
    const uint64_t bkey = mix64(seed + (base + 255 + 1) * GOLDEN);
    for (int e = tid; e < n * nrhs; e += BL_NT) {
        const double x = bl_normal_at(bkey, e);
        Bp[e] = x;
        Xp[e] = x;
    }
    __syncthreads();
    for (int pass = 0; pass < 2; ++pass) {
        for (int q = 0; q < nrefl; ++q) {
            // pass 0: U^T y = H_nrefl..H_1 y (H_1 first); pass 1: V y (H'_nrefl first)
            const int i = pass == 0 ? q : nrefl - 1 - q;
            const double vtv = bl_load_reflector(seed, base + (pass ? 128 : 0) + i, n, v, red);
            const double f = 2.0 / vtv;
            for (int c = wave; c < nrhs; c += 4) {
                double s = 0.0;
                for (int r = lane; r < n; r += 64) s += v[r] * Xp[r * nrhs + c];
                s = bl_wave_sum(s);
                if (lane == 0) w[c] = s;
            }
            __syncthreads();
            for (int e = tid; e < n * nrhs; e += BL_NT) {
                const int r = e / nrhs, c = e - r * nrhs;
                Xp[e] -= f * v[r] * w[c];
            }
            __syncthreads();
        }
        if (pass == 0) {
            for (int e = tid; e < n * nrhs; e += BL_NT) Xp[e] /= sigma(e / nrhs);
            __syncthreads();
        }
    }
}

}  // namespace lahip

using namespace lahip;

extern "C" int la_gen_svd_batch_dev(la_ctx *ctx, int64_t count, const int32_t *d_n,
                                    const int32_t *d_nrhs, const int64_t *d_offA,
                                    const int64_t *d_offB, double kappa, int nrefl, uint64_t seed,
                                    uint64_t stream_base, double *A, double *B, double *Xstar)
{
    if (!ctx || !d_n || !d_nrhs || !d_offA || !d_offB || !A || !B || !Xstar || count <= 0 ||
        count > INT32_MAX || nrefl < 0 || nrefl > 128 || !(kappa >= 1.0))
        return LA_ERR_ARG;
    hipLaunchKernelGGL(k_gen_svd_batch, dim3((unsigned)count), dim3(BL_NT), 0, ctx->stream,
                       (int)count, d_n, d_nrhs, d_offA, d_offB, kappa, nrefl, seed, stream_base, A,
                       B, Xstar);
    LA_HIP_CHECK(ctx, hipGetLastError());
    return LA_OK;
}
