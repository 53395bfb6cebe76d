// Shared by the LU kernels: block sizes, pivot keys, wavefront argmax and the
// relaxed device-scope accesses of the exchanges between workgroups.
#pragma once
#include "la_common.hpp"
#include "lu_schedule.hpp"

namespace lahip {

constexpr int PANEL_MAXP = 256;     // max cooperative workgroups in a panel

// ---------------------------------------------------------------- keys
// Ordered key for |v|: NaN -> 0 (never wins), otherwise bits(|v|)+1, so that
// unsigned comparison of keys is comparison of |v| and 0 beats NaN.
__device__ inline uint64_t abs_key(double v) {
    if (v != v) return 0;
    return (uint64_t)(__double_as_longlong(v) & 0x7fffffffffffffffLL) + 1;
}
__device__ inline uint64_t abs_key(float v) {
    if (v != v) return 0;
    return (uint64_t)(__float_as_uint(v) & 0x7fffffffu) + 1;
}
constexpr uint64_t KEY_MAX = 0x7fffffffffffffffULL;
constexpr uint64_t TAG_BIT = 0x8000000000000000ULL;
constexpr int IDX_NONE = 0x7fffffff;

__device__ inline bool better(uint64_t k1, int i1, uint64_t k0, int i0) {
    return k1 > k0 || (k1 == k0 && i1 < i0);
}

// Maximum of an unsigned value over the wavefront, by DPP row shifts and
// row broadcasts (no LDS round trip): lane 63 ends with the maximum, which
// every lane receives.
__device__ inline uint32_t wave_max_u32(uint32_t v)
{
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Wavefront argmax under better(): largest 64-bit key, lowest index among
// equal keys; every lane returns the winner.  Three DPP maxima (high key
// word, low key word among the lanes at the high maximum, complemented
// index among the lanes at the full maximum) instead of a shuffle tree.
__device__ inline void wave_argmax(uint64_t &key, int &idx) {
    const uint32_t hi = (uint32_t)(key >> 32), lo = (uint32_t)key;
    const uint32_t mhi = wave_max_u32(hi);
    const bool at_hi = hi == mhi;
    const uint32_t mlo = wave_max_u32(at_hi ? lo : 0u);
    const bool at_max = at_hi && lo == mlo;
    const uint32_t nidx = wave_max_u32(at_max ? ~(uint32_t)idx : 0u);
    key = ((uint64_t)mhi << 32) | mlo;
    idx = (int)~nidx;
}

__device__ inline uint64_t ld_relaxed(const uint64_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_relaxed(uint64_t *p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline int ld_status(const int32_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// y / d from rd = 1 / d: the product, corrected by its residual to what a
// division gives (a last bit apart where the residual is subnormal).  Not
// finite where y, d, rd or the quotient is not: there the caller divides.
__device__ inline double div_rcp(double y, double d, double rd) {
    const double q = y * rd;
    return fma(fma(-q, d, y), rd, q);
}
__device__ inline float div_rcp(float y, float d, float rd) {
    const float q = y * rd;
    return fmaf(fmaf(-q, d, y), rd, q);
}

constexpr int BLK_MAP_MAX = 2 * NB_OUT;         // rows a block's swaps can move

// A layout of the column-distributed block kernel (getrf_block.hip).
struct BlockCfg {
    int rows, cw;               // rows held, columns per workgroup
    const void *fn;
    int nt;                     // threads
    size_t lds;
};
// The layout for a block of M rows whose workgroups find num_cus CUs, or null.
template <typename T> const BlockCfg *block_cfg(int64_t M, int num_cus);
// What the block kernel needs beyond the row-distributed panels' workspace:
// published multipliers (NB_OUT columns of the tallest layout), the words that
// announce them, the swap map of a whole block.
constexpr size_t BLK_PUB_BYTES = (size_t)NB_OUT * 8192 * sizeof(double);
constexpr size_t BLK_PV_BYTES = NB_OUT * sizeof(uint64_t);
constexpr size_t BLK_MAP_BYTES = (1 + 2 * BLK_MAP_MAX) * sizeof(int64_t);
constexpr size_t BLK_SLOT_BYTES = BLK_PUB_BYTES + BLK_PV_BYTES + BLK_MAP_BYTES;

// Inverses of the 64 x 64 diagonal triangles of a packed LU of order n (unit
// lower, or upper), and X <- T^-1 X for a block of nbo <= NB_OUT rows with
// them (trsm_block.hip); refine: with one correction per 64 rows.
template <typename T>
int launch_block_inv(la_ctx *ctx, bool upper, const T *Tm, int64_t ldt, int64_t n, T *inv);
template <typename T>
int launch_trsm_block(la_ctx *ctx, bool upper, const T *Tm, int64_t ldt, const T *inv, int nbo,
                      T *B, int64_t ldb, int64_t ncols, bool refine = false);

}  // namespace lahip
