"""The LU's choice of where look-ahead starts (lu_schedule.hpp), on the host:
every block from there on is factored by a kernel whose workgroups the panel
stream's CUs hold.  The row-distributed panel is modelled by its rows per
workgroup (64, 128, 192; FP32 also 256) and two or three workgroups a CU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "lu_schedule.hpp"
#include <cstdio>
#include <initializer_list>
using namespace lahip;
static bool rows_fit(int elem, int64_t rows, int cus, int occ)
{
    for (int r = 1; r <= (elem == 8 ? 3 : 4); ++r) {
        const int64_t p = (rows + 64 * r - 1) / (64 * r);
        if (p <= 256 && p <= (int64_t)cus * occ) return true;
    }
    return false;
}
int main()
{
    long cases = 0, with = 0;
    for (int elem : {4, 8})
        for (int cus : {32, 64, 96, 128})
            for (int occ : {1, 2, 3})
                for (int64_t m = 64; m <= 40000; m += m < 600 ? 37 : 331) {
                    auto fits = [&](int64_t K0) {
                        const int wg = block_workgroups(elem, m - K0);
                        return wg ? wg <= cus : rows_fit(elem, m - K0, cus, occ);
                    };
                    for (int64_t n : {m, m / 2 + 1, m + 300}) {
                        const int64_t kmax = m < n ? m : n;
                        const int64_t from = lookahead_from(kmax, n, fits);
                        ++cases;
                        if (from == kmax) continue;
                        ++with;
                        if (from % NB_OUT || from + NB_OUT >= kmax || from + NB_OUT >= n) return 1;
                        for (int64_t K0 = from; K0 < kmax; K0 += NB_OUT)
                            if (!fits(K0)) {
                                printf("elem %d cus %d occ %d m %ld n %ld: from %ld, block %ld\n", elem,
                                       cus, occ, (long)m, (long)n, (long)from, (long)K0);
                                return 1;
                            }
                        if (from > 0 && fits(from - NB_OUT)) return 1;
                    }
                }
    printf("%ld of %ld\n", with, cases);
    return with > 0 ? 0 : 1;
}
"""


def test_lookahead_start(tmp_path):
    src = tmp_path / "schedule.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "schedule"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I",
                    os.path.join(ROOT, "rust-la_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
