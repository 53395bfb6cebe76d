// Choices of the blocked LU that depend on sizes alone, with no device code:
// the layouts of the column-distributed block and the outer block from which
// the look-ahead schedule can run.
#pragma once
#include <stdint.h>

namespace lahip {

constexpr int NB_IN = 64;           // inner panel width
constexpr int NB_OUT = 256;         // outer block width (trailing GEMM K)

// A layout holds `rows` rows and gives each workgroup `cw` columns.
struct BlockShape { int rows, cw; };
constexpr BlockShape BLOCK_SHAPES_F64[] = {{512, 32}, {1024, 16}, {2048, 16}, {4096, 8}, {8192, 4}};
constexpr BlockShape BLOCK_SHAPES_F32[] = {{512, 32}, {1024, 32}, {2048, 32},
                                           {4096, 16}, {8192, 8}, {16384, 4}};
// Workgroups of the layout that takes an outer block of `rows` rows, all of
// which have to be resident at once; 0 if it is too tall.
inline int block_workgroups(int elem, int64_t rows)
{
    if (elem == 8) {
        for (const BlockShape &s : BLOCK_SHAPES_F64)
            if (rows <= s.rows) return NB_OUT / s.cw;
    } else {
        for (const BlockShape &s : BLOCK_SHAPES_F32)
            if (rows <= s.rows) return NB_OUT / s.cw;
    }
    return 0;
}

// First column of the outer block from which look-ahead can run: the kernel
// that factors each block from there to the last fits the panel stream
// (fits(K0); not only the first one, since a shorter block may go to a kernel
// that needs more CUs), and there are columns to look ahead to.  kmax if none.
template <typename Fits>
int64_t lookahead_from(int64_t kmax, int64_t n, Fits fits)
{
    int64_t from = 0;
    for (int64_t K0 = 0; K0 < kmax; K0 += NB_OUT)
        if (!fits(K0)) from = K0 + NB_OUT;
    return from + NB_OUT < kmax && from + NB_OUT < n ? from : kmax;
}

}  // namespace lahip
