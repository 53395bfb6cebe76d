// The column-distributed outer block of the LU factorisation: every column of
// a block of up to 256 in one launch (k_getrf_block).
#include "lu_device.hpp"
#include <utility>

namespace lahip {

// ------------------------------------------------- column-distributed block
// Factors a whole outer block (M rows x nbo <= NB_OUT columns, top-left
// element A) in ONE launch.  Workgroup g owns columns [g CW, (g+1) CW) of
// ALL rows and keeps them in registers from the first load to the final
// store: thread t holds rows t + NT q, q < RPT.  So the pivot search, the
// multipliers and the rank-1 updates of a workgroup's CW columns stay on one
// CU (one barrier per column), and workgroups exchange once per column in
// one direction only: the owner publishes column k's multipliers (every row,
// in row order) and its pivot row; every workgroup to the right applies them
// to its own columns while the owner goes on.  The row-distributed panel
// (k_getrf_panel) instead crosses CUs twice per column on the critical path.
//
// Rows never move: s_pos[r] is row r's current position, s_inv[p] the row at
// position p < nbo, and a pivot swap relabels two rows in every workgroup.
// A row that becomes pivot k is final in columns right of k: its owner
// stores the workgroup's CW values of it in s_u[k].  Its multiplier is
// published as 1, so the update with itself leaves exact zeros in the owner's
// registers (the workgroups to the right store zeros): its later multipliers
// are zero, it can never win a pivot search and the updates need no per-row
// condition.  At the end each row goes to its final position, from s_u if it
// was a pivot up to this workgroup's last column and from the registers (its
// multipliers) if not.
//
// Pivot rule: largest |v|, lowest position on ties, a NaN never preferred
// over a number and kept if it sits at position j (lu.rs:132-137).  The
// search compares the high (FP32: only) word of |v| without its lowest
// log2(RPT) bits, which name the row's register; it is decided when one row
// alone holds the maximum, finite and not zero.  Anything else (a second row
// that close, a zero column, Inf or NaN) takes the full-key search over the
// positions.
//
// The columns to the left are applied LB at a time, their products summed
// first and then taken from the element: one after the other they rounded
// every element up to 255 times, and the error of an FP32 factor of n = 16384
// with singular values in [1e-6, 1] was 1.6 times that of 64-column panels with
// GEMM updates between them (now 0.6 times; the batches cost 2-9% of a
// factorisation).  The batch is fixed, not what happens to be published, so
// that a factor does not depend on timing.  Its pivot rows, as they stand
// before it, are brought up to date by a triangular solve of order LB.
//
// Exchange: column k's multipliers go out with device-coherent stores, every
// wave waits for its own, and after the next barrier one thread stores the
// word pv[k] = (kglob + k) << 32 | pivot row.  A consumer reads multipliers
// only after it saw pv[k], and a published column does not change, so its
// caches cannot hold an older copy (they are invalidated between launches) and
// plain loads, shared by the workgroups of an XCD through its L2, suffice.  pv is
// reset once per factorisation: each kglob + k occurs once in it.  Every
// wait is bounded and ends all workgroups through `status`.
//
// Bound by latency: per column one barrier, the wave and workgroup maxima,
// the reciprocal and the LDS reads of the pivot row; per CW columns the
// hand-over to the next workgroup (a store's way to memory, the poll, the
// load of the multipliers).  Measured on the panel stream, 256 columns:
// FP64 920 us at 4096-8192 rows (767 with the left columns applied one at a
// time), 560 at 2048-4096, 590 at 1024-2048, 480 below; FP32 1040 at 8192-16384
// (888), 645 at 1024-8192, 500 at 512-1024, 390 below.  Four row-distributed
// panels with their in-block row moves, TRSM and GEMM took 1.1-1.5 ms.
//
// Layout: NT x RPT rows and CW columns so that a thread's RPT x CW elements
// take 128 registers (64 for the smallest): fewer, taller threads spend less
// on the per-wave part of a column (wave maximum, candidate read,
// reciprocal), and a wider CW amortises the hand-over between workgroups.
template <typename F, int... I>
__device__ __forceinline__ void for_each_index(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <typename T> struct AbsWord;
template <> struct AbsWord<double> {
    static constexpr uint32_t INF = 0x7ff00000u;
    __device__ static inline uint32_t of(double v) {
        return (uint32_t)((uint64_t)__double_as_longlong(v) >> 32) & 0x7fffffffu;
    }
};
template <> struct AbsWord<float> {
    static constexpr uint32_t INF = 0x7f800000u;
    __device__ static inline uint32_t of(float v) { return __float_as_uint(v) & 0x7fffffffu; }
};

template <typename T, int NT, int RPT, int CW> struct BlockLds {
    static constexpr int NW = NT / 64;
    T u[NB_OUT * CW];                   // pivot rows, this workgroup's columns
    T crow[2][NW][CW];                  // candidate rows by step parity and wave
    T srow[CW];                         // winner row of a full-key search
    T lp[8][8];                         // multipliers of a batch's pivot rows
    uint64_t skey[NW];
    int sidx[NW], swin;
    uint32_t cval[2][NW];
    int cid[2][NW];
    int prow[NB_OUT];                   // pivot row of each column seen so far
    int avail, abort, nmoves;
    uint16_t pos[NT * RPT];
    uint16_t inv[NB_OUT];
};

template <typename T, int NT, int RPT, int CW>
__global__ __launch_bounds__(NT)
void k_getrf_block(T *A, int64_t lda, int M, int nbo, int kglob, int64_t *ipiv, T *pub,
                   uint64_t *pv, int64_t *swapmap, int32_t *status, uint64_t spin_ticks)
{
    constexpr int NW = NT / 64, UN = CW < 8 ? CW : 8, NBLK = CW / UN;
    // columns of the left workgroups applied together, and the rows of their
    // multipliers held at a time: 32 registers in FP64, 64 in FP32 (64 in FP64
    // made n = 8192 1.5% slower, 32 in FP32 n = 16384 0.8%)
    constexpr int LB = CW >= 32 ? 8 : 4;
    constexpr int QF = (sizeof(T) == 8 ? 16 : 64) / LB, QG = QF < RPT ? QF : RPT;
    // multipliers as quotients in the lowest layout, as k_getrf_panel_local's;
    // products with the pivot's reciprocal above, as k_getrf_panel's
    constexpr bool QUOT = NT * RPT <= 512;
    constexpr int64_t LDP = NT * RPT;
    typedef T vr __attribute__((ext_vector_type(RPT)));
    extern __shared__ __align__(16) unsigned char blk_smem[];
    BlockLds<T, NT, RPT, CW> &S = *reinterpret_cast<BlockLds<T, NT, RPT, CW> *>(blk_smem);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = blockIdx.x, col0 = g * CW;
    const int ncol = min(CW, nbo - col0);               // >= 1 by the grid

    // a[i][q]: column i of row tid + NT q.  One register vector per column:
    // a row picked at run time (q the same in the whole wave) is an indexed
    // register read, not a branch per row.
    vr a[CW];
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const int r = tid + NT * q;
        const T *src = A + (int64_t)min(r, M - 1) * lda + col0;
#pragma unroll
        for (int i = 0; i < CW; ++i) a[i][q] = src[min(i, ncol - 1)];
    }
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const int r = tid + NT * q;
#pragma unroll
        for (int i = 0; i < CW; ++i) a[i][q] = r < M && i < ncol ? a[i][q] : T(0);
        S.pos[r] = (uint16_t)r;
    }
    for (int i = tid; i < NB_OUT; i += NT) S.inv[i] = (uint16_t)i;
    if (tid == 0) { S.abort = 0; S.nmoves = 0; }
    // a wait that is given up leaves no rows to move
    if (g == 0 && tid == 0) swapmap[0] = 0;

    // swap of position k with the position of row rp (one thread); returns
    // that position
    auto relabel = [&](int k, int rp) __attribute__((always_inline)) -> int {
        const int p = S.pos[rp];
        if (p != k) {
            const int rj = S.inv[k];
            S.pos[rj] = (uint16_t)p;
            S.pos[rp] = (uint16_t)k;
            S.inv[k] = (uint16_t)rp;
            if (p < NB_OUT) S.inv[p] = (uint16_t)rj;
        }
        return p;
    };
    // wave 0: waits until column k is published; notes the pivot rows of it
    // and of the columns after it that are published too (at most to kend).
    // Returns the first column not yet seen, or -1 when the wait is given up.
    auto poll = [&](int k, int kend) __attribute__((always_inline)) -> int {
        const int idx = min(k + lane, kend - 1);
        const uint64_t *src = pv + idx;
        const uint64_t t0 = wall_clock64();
        for (uint32_t spin = 0;; ++spin) {
            const uint64_t w = ld_relaxed(src);
            const bool ok = (uint32_t)(w >> 32) == (uint32_t)(kglob + idx);
            const uint64_t bal = __ballot(ok);
            if (bal & 1) {
                const int n = min(~bal ? __ffsll((unsigned long long)~bal) - 1 : 64, kend - k);
                if (lane < n) S.prow[k + lane] = min((int)(uint32_t)w, M - 1);
                return k + n;
            }
            if ((spin & 31) == 31 && ld_status(status) != 0) return -1;
            if (wall_clock64() - t0 > spin_ticks) {
                if (lane == 0) atomicCAS((int *)status, 0, (int)LA_ERR_TIMEOUT);
                return -1;
            }
            __builtin_amdgcn_s_sleep(1);
        }
    };
    // row rk's values, from its owner's registers (rotated by `it` blocks),
    // in column order to dst (LDS)
    auto put_row = [&](T *dst, int rk, int it) __attribute__((always_inline)) {
        const int qo = __builtin_amdgcn_readfirstlane(rk / NT);
        if (wave == (rk & (NT - 1)) >> 6) {
            T v[CW];
#pragma unroll
            for (int i = 0; i < CW; ++i) v[i] = a[i][qo];
            if (tid == (rk & (NT - 1))) {
#pragma unroll
                for (int b = 0; b < NBLK; ++b)
#pragma unroll
                    for (int i = 0; i < UN; ++i) dst[((b + it) % NBLK) * UN + i] = v[b * UN + i];
            }
        }
    };

    __syncthreads();

    // ---- the columns to the left, LB at a time: a -= sum of l u
    for (int k = 0, avail = 0; k < col0; k += LB) {
        while (avail < k + LB) {                        // uniform
            if (wave == 0) {
                const int v = poll(avail, col0);
                if (lane == 0) S.avail = v;
            }
            __syncthreads();
            avail = __builtin_amdgcn_readfirstlane(S.avail);
            if (avail < 0) return;                      // every wave
            __syncthreads();
        }
        // the batch's pivot rows as they stand before it, and their
        // multipliers in its columns
#pragma unroll 1
        for (int b = 0; b < LB; ++b)
            put_row(S.u + (k + b) * CW, __builtin_amdgcn_readfirstlane(S.prow[k + b]), 0);
        if (tid < LB * LB)
            S.lp[tid / LB][tid % LB] = pub[(int64_t)(k + tid % LB) * LDP + S.prow[k + tid / LB]];
        if (tid == NT - 1)
            for (int b = 0; b < LB; ++b) relabel(k + b, S.prow[k + b]);
        __syncthreads();
        // u_b = a_b - sum_{c<b} l_bc u_c, one column per lane
        if (tid < CW) {
            T u[LB];
#pragma unroll
            for (int b = 0; b < LB; ++b) {
                u[b] = S.u[(k + b) * CW + tid];
#pragma unroll
                for (int c = 0; c < b; ++c) u[b] -= S.lp[b][c] * u[c];
                S.u[(k + b) * CW + tid] = u[b];
            }
        }
        __syncthreads();
#pragma unroll
        for (int q0 = 0; q0 < RPT; q0 += QG) {
            // one group's loads at a time, u read again for each
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("" ::: "memory");
            T l[LB][QG];
#pragma unroll
            for (int b = 0; b < LB; ++b) {
                const T *src = pub + (int64_t)(k + b) * LDP + NT * q0;
#pragma unroll
                for (int q = 0; q < QG; ++q) l[b][q] = (src + NT * q)[(uint32_t)tid];
            }
#pragma unroll
            for (int i = 0; i < CW; ++i) {
                T u[LB];
#pragma unroll
                for (int b = 0; b < LB; ++b) u[b] = S.u[(k + b) * CW + i];
#pragma unroll
                for (int q = 0; q < QG; ++q) {
                    T d = l[0][q] * u[0];
#pragma unroll
                    for (int b = 1; b < LB; ++b) d += l[b][q] * u[b];
                    a[i][q0 + q] -= d;
                }
            }
        }
        // the pivot rows are final: exact zeros in the registers
#pragma unroll 1
        for (int b = 0; b < LB; ++b) {
            const int rk = __builtin_amdgcn_readfirstlane(S.prow[k + b]);
            const int qo = __builtin_amdgcn_readfirstlane(rk / NT);
            if (wave == (rk & (NT - 1)) >> 6) {
                const bool mine = tid == (rk & (NT - 1));
#pragma unroll
                for (int i = 0; i < CW; ++i) {
                    const T v = a[i][qo];
                    a[i][qo] = mine ? T(0) : v;
                }
            }
        }
    }

    // ---- this workgroup's own columns.  The column being eliminated is
    // register s of the current block of UN; after UN columns the registers
    // rotate by one block, so the loop body is UN columns long, not CW.
    auto column = [&](auto s_c, int it) __attribute__((always_inline)) {
            constexpr int s = decltype(s_c)::value;
            const int c = it * UN + s;
            if (c >= ncol) return;                      // uniform
            const int j = col0 + c, par = c & 1;
            // wave candidate: the high word of |v| with the row's register
            // index in its lowest bits; m2 the second largest
            uint32_t m = 0, m2 = 0;
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const uint32_t k = (AbsWord<T>::of(a[s][q]) & ~(uint32_t)(RPT - 1)) | q;
                m2 = max(min(k, m), m2);
                m = max(m, k);
            }
            const uint32_t wm = wave_max_u32(m);
            const uint64_t whit = __ballot(m == wm);
            const int wl = __ffsll((unsigned long long)whit) - 1;
            // another row in the winner's bucket: this wave cannot decide
            const bool tied = __any((m2 | (RPT - 1)) == (wm | (RPT - 1))) ||
                              __popcll(__ballot((m | (RPT - 1)) == (wm | (RPT - 1)))) != 1;
            const int wrow = wave * 64 + wl + NT * (int)(wm & (RPT - 1));
            put_row(S.crow[par][wave], wrow, it);
            if (lane == 0) {
                S.cval[par][wave] = wm | (RPT - 1);
                S.cid[par][wave] = wrow | (tied ? 1 << 30 : 0);
            }
            // the previous column's multipliers have left this wave
            stores_done();
            __syncthreads();
            if (tid == 64 && c > 0)
                st_relaxed(pv + j - 1, ((uint64_t)(uint32_t)(kglob + j - 1) << 32) |
                                           (uint32_t)S.prow[j - 1]);
            const uint32_t cv = S.cval[par][lane & (NW - 1)];
            const uint32_t gm = wave_max_u32(cv);
            const uint64_t win = __ballot(cv == gm) & ((1ull << NW) - 1);
            const int ww = __ffsll((unsigned long long)win) - 1;
            const T *urow = S.crow[par][ww];
            int rp = __builtin_amdgcn_readfirstlane(S.cid[par][ww]);
            if (gm < RPT || gm >= AbsWord<T>::INF || __popcll(win) != 1 || (rp >> 30)) {
                // full-key search over the rows at positions >= j
                uint64_t key = 0;
                int idx = IDX_NONE;
#pragma unroll
                for (int q = 0; q < RPT; ++q) {
                    const int r = tid + NT * q;
                    const int p = S.pos[r];
                    if (r < M && p >= j) {
                        const T v = a[s][q];
                        uint64_t k = abs_key(v);
                        if (p == j && v != v) k = KEY_MAX;
                        if (better(k, p, key, idx)) { key = k; idx = p; }
                    }
                }
                wave_argmax(key, idx);
                if (lane == 0) { S.skey[wave] = key; S.sidx[wave] = idx; }
                __syncthreads();
                key = S.skey[0];
                idx = S.sidx[0];
                for (int w = 1; w < NW; ++w)
                    if (better(S.skey[w], S.sidx[w], key, idx)) { key = S.skey[w]; idx = S.sidx[w]; }
                for (int r = tid; r < M; r += NT)
                    if (S.pos[r] == idx) S.swin = r;
                __syncthreads();
                rp = __builtin_amdgcn_readfirstlane(S.swin);
                put_row(S.srow, rp, it);
                __syncthreads();
                urow = S.srow;
            }
            T u[CW];                                    // in register order
#pragma unroll
            for (int b = 0; b < NBLK; ++b) {
                const T *src = urow + ((b + it) % NBLK) * UN;
#pragma unroll
                for (int i = 0; i < UN; ++i) u[b * UN + i] = src[i];
            }
            if (tid < CW) S.u[j * CW + tid] = urow[tid];
            if (tid == 64) {
                S.prow[j] = rp;
                ipiv[kglob + j] = (int64_t)kglob + relabel(j, rp);
            }
            const T piv = u[s];
            const T rpiv = piv != T(0) ? T(1) / piv : T(1);
            const bool fin = AbsWord<T>::of(rpiv) < AbsWord<T>::INF &&
                             AbsWord<T>::of(piv) < AbsWord<T>::INF;
            vr l;
            if (fin) {
                if constexpr (QUOT) {
                    // a zero pivot leaves the column as it is
                    const T d = piv != T(0) ? piv : T(1);
#pragma unroll
                    for (int q = 0; q < RPT; ++q) l[q] = div_rcp((T)a[s][q], d, rpiv);
                } else {
                    l = a[s] * (vr)rpiv;
                }
            } else {
                // the pivot is infinite or a NaN, or its reciprocal overflows:
                // divide, and keep the rows that are already final out of it
                __syncthreads();                        // positions of this step
#pragma unroll
                for (int q = 0; q < RPT; ++q) {
                    const int r = tid + NT * q;
                    l[q] = (r < M && S.pos[r] > j) ? a[s][q] / piv : T(0);
                }
            }
            // the pivot row's own multiplier is 1: its update leaves exact
            // zeros, here and in the workgroups to the right
            if (wave == ((rp & (NT - 1)) >> 6)) {
                const int d = rp - tid;
#pragma unroll
                for (int q = 0; q < RPT; ++q)
                    if (d == NT * q) l[q] = T(1);
            }
            T *dst = pub + (int64_t)j * LDP;
#pragma unroll
            for (int q = 0; q < RPT; ++q) st_dev(dst + NT * q + (uint32_t)tid, (T)l[q]);
            a[s] = l;
            // the columns right of c: the register blocks past NBLK - it
            // hold finished columns again
#pragma unroll
            for (int b = 0; b < NBLK; ++b)
                if (b < NBLK - it) {
#pragma unroll
                    for (int i = 0; i < UN; ++i)
                        if (b * UN + i > s) a[b * UN + i] -= l * (vr)u[b * UN + i];
                }
    };
    for (int it = 0; it < NBLK; ++it) {
        for_each_index([&](auto s_c) __attribute__((always_inline)) { column(s_c, it); },
                       std::make_integer_sequence<int, UN>{});
        if (NBLK > 1) {
            vr t[UN];
#pragma unroll
            for (int i = 0; i < UN; ++i) t[i] = a[i];
#pragma unroll
            for (int i = 0; i < CW - UN; ++i) a[i] = a[i + UN];
#pragma unroll
            for (int i = 0; i < UN; ++i) a[CW - UN + i] = t[i];
        }
    }
    stores_done();
    __syncthreads();
    const int kown = col0 + ncol;               // this workgroup's last column + 1
    if (tid == 64)
        st_relaxed(pv + kown - 1, ((uint64_t)(uint32_t)(kglob + kown - 1) << 32) |
                                      (uint32_t)S.prow[kown - 1]);

    // ---- the pivots of the columns to the right, for the final positions
    if (wave == 0) {
        int k = kown;
        while (k < nbo) {
            const int v = poll(k, nbo);
            if (v < 0) { if (lane == 0) S.abort = 1; break; }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            if (lane == 0)
                for (; k < v; ++k) relabel(k, S.prow[k]);
            k = v;
        }
    }
    __syncthreads();
    if (S.abort) return;
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const int r = tid + NT * q;
        if (r < M) {
            const int p = S.pos[r];
            T *dst = A + (int64_t)p * lda + col0;
            const bool done = p < kown;
#pragma unroll
            for (int i = 0; i < CW; ++i) {
                const T v = done ? S.u[p * CW + i] : (T)a[i][q];
                if (i < ncol) dst[i] = v;
            }
            if (g == 0 && p != r) {
                const int e = atomicAdd(&S.nmoves, 1);
                swapmap[1 + 2 * e] = (int64_t)kglob + p;
                swapmap[2 + 2 * e] = (int64_t)kglob + r;
            }
        }
    }
    if (g == 0) {
        __syncthreads();
        if (tid == 0) swapmap[0] = S.nmoves;
    }
}

// ------------------------------------------- column-distributed block: host
// Layouts of k_getrf_block by rows, in order of height.  The first that
// holds M rows is taken.  Rows x columns per workgroup fill 128 registers a
// thread; past the tallest the row-distributed panels run (two columns per
// workgroup would hand over on every second column).
template <typename T, int I, int NT, int RPT> static BlockCfg block_cfg_of()
{
    constexpr BlockShape s = sizeof(T) == 8 ? BLOCK_SHAPES_F64[I < 5 ? I : 0] : BLOCK_SHAPES_F32[I];
    static_assert(s.rows == NT * RPT, "rows of the layout");
    return BlockCfg{s.rows, s.cw, (const void *)k_getrf_block<T, NT, RPT, s.cw>, NT,
                    sizeof(BlockLds<T, NT, RPT, s.cw>)};
}
template <typename T> const BlockCfg *block_cfg(int64_t M, int num_cus)
{
    static const std::vector<BlockCfg> cfgs = [] {
        std::vector<BlockCfg> v = {block_cfg_of<T, 0, 256, 2>(), block_cfg_of<T, 1, 256, 4>(),
                                   block_cfg_of<T, 2, 512, 4>(), block_cfg_of<T, 3, 512, 8>(),
                                   block_cfg_of<T, 4, 512, 16>()};
        if constexpr (sizeof(T) == 4) v.push_back(block_cfg_of<T, 5, 512, 32>());
        for (auto &c : v)
            if (c.lds > allow_dynamic_lds(c.fn)) c.rows = 0;
        return v;
    }();
    for (const auto &c : cfgs)
        if (M <= c.rows && NB_OUT / c.cw <= num_cus) return &c;
    return nullptr;
}
static_assert(BLK_PUB_BYTES >= (size_t)NB_OUT * 16384 * sizeof(float), "tallest layouts");

template const BlockCfg *block_cfg<double>(int64_t, int);
template const BlockCfg *block_cfg<float>(int64_t, int);


}  // namespace lahip
