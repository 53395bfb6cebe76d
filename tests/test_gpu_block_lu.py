"""The column-distributed outer block of the LU (getrf_block.hip) where it can
go wrong: the row counts at which its register layouts change (512, 1024,
2048, 4096, 8192 rows in FP64), widths that leave the last workgroup or the
last block ragged, and pivot searches that the high word of |v| cannot decide
(ties, zero columns, NaN, Inf) against LUDecomposition::new
(src/decomp/lu.rs:104-168)."""
import numpy as np
import pytest

import la_hip
import oracle

pytestmark = pytest.mark.gpu


def _pivots(ctx, a):
    lu, piv, sign = ctx.lu_new(a)
    lu_o, piv_o, sign_o = oracle.lu_new(a)
    assert np.array_equal(piv, piv_o) and sign == sign_o
    return lu, lu_o


# factors within 1e-10 of the oracle's, as the parity tests of the other sizes
@pytest.mark.parametrize("shape", [(512, 257), (513, 70), (1024, 97), (1025, 256), (2048, 129),
                                   (2049, 65), (4096, 72), (4097, 260), (8192, 68), (8193, 67),
                                   (190, 190), (300, 800)])
def test_layout_edges(ctx, shape):
    a = oracle.uniform(31, shape[0] + shape[1], shape)
    lu, lu_o = _pivots(ctx, a)
    assert np.abs(lu - lu_o).max() <= 1e-10 * np.abs(lu_o).max()


# One non-zero per row, a power of two: every elimination step is exact, so
# the pivots and the factor are the oracle's bit for bit, ties included.
@pytest.mark.parametrize("m,n", [(400, 300), (1100, 100), (5000, 80)])
def test_ties_and_zero_columns(ctx, m, n):
    rng = np.random.default_rng(m)
    a = np.zeros((m, n))
    rows = np.arange(m)
    a[rows, rng.permutation(rows) % n] = rng.choice([-2.0, -1.0, 1.0, 2.0], size=m)
    a[:, rng.permutation(n)[:5]] = 0.0
    lu, lu_o = _pivots(ctx, a)
    assert np.array_equal(lu, lu_o)


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("m,row,col", [(300, 40, 40), (300, 100, 40), (2500, 66, 66),
                                       (2500, 2400, 3)])
def test_nan_and_inf(ctx, m, row, col, bad):
    a = oracle.uniform(77, m, (m, 90))
    a[row, col] = bad
    lu, lu_o = _pivots(ctx, a)
    assert np.array_equal(np.isnan(lu), np.isnan(lu_o))


# FP32 layouts: 512, 1024, 2048, 4096 and 8192 rows and one more
@pytest.mark.parametrize("n", [512, 513, 1025, 2049, 4097, 8193])
def test_fp32_layout_edges(tctx, torch_cuda, n):
    torch = torch_cuda
    A = torch.empty((n, n), dtype=torch.float64, device="cuda")
    b = torch.empty((n, 1), dtype=torch.float64, device="cuda")
    tctx.gen_svd_matrix_dev(n, 1e3, 8, 5, A, b=b, xstar=torch.empty_like(b))
    X = torch.empty_like(b)
    rep = tctx.gesv_ir_dev(A, b, X, la_hip.PREC_FP32, 1e-15 * n, 30)
    torch.cuda.synchronize()
    r = (b - A @ X).abs().max().item()
    eta = r / (A.abs().sum(1).max().item() * X.abs().max().item() + b.abs().max().item())
    # FP32 factor at kappa 1e3: one correction contracts the error by about
    # kappa * n * 2^-24 * growth << 1, so a second one reaches FP64 accuracy
    assert rep.status == la_hip.LA_OK and rep.iterations <= 3
    assert eta <= 1e-15 * n


# Roundings per element: with pivots of 2^20, multipliers near 2^-20 and
# elements that stay in [1, 2), each subtraction rounds an element by up to
# half of 2^-52, independent of the others.  A column c of the block sees the
# sums of four or more columns from the workgroups to its left and at most cw
# single ones of its own; the quotient, the multiplier's own rounding and the
# sums add less than four more.  (Column by column it would be c: 2.5 to 4
# times the bound.)
@pytest.mark.parametrize("m,cw", [(400, 32), (900, 16), (3000, 8), (5000, 4)])
def test_roundings_per_element(tctx, torch_cuda, m, cw):
    torch, n = torch_cuda, 256
    rng = np.random.default_rng(m)
    a = rng.uniform(1.25, 1.75, (m, n))
    a[np.arange(n), np.arange(n)] = 2.0 ** 20
    W = torch.from_numpy(a).cuda()
    piv = torch.empty(m, dtype=torch.int64, device="cuda")
    info = torch.zeros(4, dtype=torch.int32, device="cuda")
    tctx.getrf_dev(W, piv, info)
    assert info[1].item() == 0 and torch.equal(piv.cpu(), torch.arange(m))
    lu = W.cpu().numpy().astype(np.longdouble)
    l, u = np.tril(lu, -1)[n:], np.triu(lu[:n])
    c = np.arange(192, 256)
    r = a[n:, c] - l @ u[:, c]
    assert ((r ** 2).mean(0) <= (c / 4 + cw + 4) * 2.0 ** -104 / 12 * 1.25).all()
