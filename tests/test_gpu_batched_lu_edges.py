"""The batched LU (batched_lu.hip) at the edges of its blocks: 8-column panel
blocks, 16/32-column panels, 64-row outer and solve blocks, 256-column chunks,
and pivot searches full of ties."""
import numpy as np
import pytest

import la_hip
from test_gpu_batched_lu import eta_of, host_problem, make_batch, solve_batch

pytestmark = pytest.mark.gpu

PRECS = [la_hip.PREC_FP64, la_hip.PREC_FP32, la_hip.PREC_FP16]


@pytest.mark.parametrize("prec", PRECS)
def test_block_edges(tctx, torch_cuda, prec):
    torch = torch_cuda
    sizes = [8, 9, 15, 24, 63, 95, 96, 97, 127, 191, 193, 255, 257, 319, 321, 511, 513, 1023, 1024]
    nrhs = [8 - i % 8 for i in range(len(sizes))]
    bt = make_batch(torch, tctx, sizes, nrhs, kappa=1e2, nrefl=16)
    (x, st, it, be), = solve_batch(torch, tctx, bt, prec, tol=1e-14)
    assert (st == 0).all(), st
    a, b = bt["A"].cpu().numpy(), bt["B"].cpu().numpy()
    for i, (n, r) in enumerate(zip(sizes, nrhs)):
        ai, bi = host_problem(bt, a, b, i)
        xi = x[bt["offB"][i]:bt["offB"][i] + n * r].reshape(n, r)
        # refined: the tolerance asked for; FP64: 4 n u, partial pivoting's
        # bound 3 n u (growth 1 on these orthogonally mixed matrices) plus
        # the residual's own rounding
        bound = 4 * n * 2.0 ** -53 + 1e-15 if prec == la_hip.PREC_FP64 else 1e-14
        assert eta_of(ai, xi, bi) <= bound, (i, n)


# One entry per row and column, a power of two: whole columns tie at zero, and
# every step is exact, so the solution is too, in each working precision.
@pytest.mark.parametrize("prec", PRECS)
def test_scaled_permutations_are_exact(tctx, torch_cuda, prec):
    torch = torch_cuda
    rng = np.random.default_rng(3)
    sizes, nrhs = [1, 17, 64, 80, 150, 300], [1, 2, 8, 5, 3, 4]
    bt = make_batch(torch, tctx, sizes, nrhs)
    a, b = np.zeros(bt["A"].numel()), np.empty(bt["B"].numel())
    want = np.empty_like(b)
    for i, (n, r) in enumerate(zip(sizes, nrhs)):
        p, d = rng.permutation(n), rng.choice([-4.0, -1.0, 0.5, 2.0], size=n)
        ai, bi = host_problem(bt, a, b, i)
        ai[np.arange(n), p] = d
        bi[:] = rng.integers(-8, 9, size=(n, r))
        want[bt["offB"][i]:bt["offB"][i] + n * r].reshape(n, r)[p] = bi / d[:, None]
    bt["A"].copy_(torch.from_numpy(a))
    bt["B"].copy_(torch.from_numpy(b))
    (x, st, it, be), = solve_batch(torch, tctx, bt, prec)
    assert (st == 0).all() and np.array_equal(x, want) and (be == 0).all()


def _solve_list(torch, ctx, prec, problems):
    sizes, nrhs = [a.shape[0] for a, _ in problems], [b.shape[1] for _, b in problems]
    bt = make_batch(torch, ctx, sizes, nrhs)
    bt["A"].copy_(torch.from_numpy(np.concatenate([a.ravel() for a, _ in problems])))
    bt["B"].copy_(torch.from_numpy(np.concatenate([b.ravel() for _, b in problems])))
    (x, st, it, be), = solve_batch(torch, ctx, bt, prec)
    return [x[o:o + n * r].reshape(n, r) for o, n, r in zip(bt["offB"], sizes, nrhs)], st, be


# Columns of very different scales: u / d of the back substitution is outside
# the range of the working precision where u x and the quotients are ordinary.
@pytest.mark.parametrize("prec,small,large", [(la_hip.PREC_FP64, 1e-160, 1e160),
                                              (la_hip.PREC_FP32, 1e-25, 1e15),
                                              (la_hip.PREC_FP16, 1e-25, 1e15)])
def test_back_substitution_range(tctx, torch_cuda, prec, small, large):
    a = np.array([[small, large], [0.0, 1.0]])
    t = 1e-5 * small                        # x = [1 - 1e-5 large, t]
    (x, y), st, be = _solve_list(torch_cuda, tctx, prec, [(a, np.array([[small], [0.0]])),
                                                          (a, np.array([[small], [t]]))])
    assert (st == 0).all() and np.array_equal(x, [[1.0], [0.0]])
    # two roundings of each operand and one per operation in working precision
    u = 2.0 ** -53 if prec == la_hip.PREC_FP64 else 2.0 ** -24
    want = np.array([[1.0 - 1e-5 * large], [t]])
    assert np.abs(y / want - 1.0).max() <= 8 * u


@pytest.mark.parametrize("prec,n,s", [(la_hip.PREC_FP64, 70, 160), (la_hip.PREC_FP32, 70, 20),
                                      (la_hip.PREC_FP16, 24, 20)])
def test_column_scales(tctx, torch_cuda, prec, n, s):
    rng = np.random.default_rng(n)
    r = rng.uniform(-1.0, 1.0, (n, n)) + 4 * np.sqrt(n) * np.eye(n)
    scale = np.where(rng.random(n) < 0.5, 10.0 ** -s, 10.0 ** s)
    b = rng.uniform(-1.0, 1.0, (n, 3))
    (x,), st, be = _solve_list(torch_cuda, tctx, prec, [(r * scale, b)])
    assert (st == 0).all()
    want = np.linalg.solve(r, b)
    # kappa_inf(r) < 6 and growth 1: at most 3 n u kappa for one solve
    u = 2.0 ** -53 if prec == la_hip.PREC_FP64 else 2.0 ** -24
    assert np.abs(x * scale[:, None] - want).max() <= 18 * n * u * np.abs(want).max()


# A NaN is no small residual: eta is not 0, and refinement does not converge.
@pytest.mark.parametrize("prec", PRECS)
def test_nan_right_hand_side(tctx, torch_cuda, prec):
    rng = np.random.default_rng(1)
    a = rng.uniform(-1.0, 1.0, (40, 40)) + 8 * np.eye(40)
    b = rng.uniform(-1.0, 1.0, (40, 2))
    bad = b.copy()
    bad[7, 1] = np.nan
    (x, y), st, be = _solve_list(torch_cuda, tctx, prec, [(a, bad), (a, b)])
    assert be[0] > 1.0 and be[1] <= 1e-14
    assert st[0] == (0 if prec == la_hip.PREC_FP64 else la_hip.LA_NOT_CONVERGED) and st[1] == 0
    assert eta_of(a, y, b) <= 1e-14


# The true residual of a converged refinement is the rounding of x and of the
# residual's own sum.  Terms of variance s, roundings independent and of
# variance at most u^2 / 3 of the partial sums: n / 4 sums of 4 (n / 4 * 10),
# two levels of pairs (2 n), four chains of n / 64 sixteens (n^2 / 128), two
# levels of pairs (2 n), and x (n).  Four chains of n / 4 terms would be
# n^2 / 8 in place of n^2 / 128: 2.5 times as far off.
def test_residual_rounding(tctx, torch_cuda):
    n, g, count = 1024, 8, 4
    bt = make_batch(torch_cuda, tctx, [n] * count, [g] * count, kappa=10, nrefl=64)
    (x, st, it, be), = solve_batch(torch_cuda, tctx, bt, la_hip.PREC_FP32, tol=0.0, max_iter=4)
    a, b = bt["A"].cpu().numpy(), bt["B"].cpu().numpy()
    for i in range(count):
        ai, bi = (v.astype(np.longdouble) for v in host_problem(bt, a, b, i))
        xi = x[bt["offB"][i]:bt["offB"][i] + n * g].reshape(n, g).astype(np.longdouble)
        s = ((ai ** 2) @ (xi ** 2)).mean() / n
        var = (n / 4 * 10 + 4 * n + n * n / 128 + n) * s * 2.0 ** -106 / 3
        assert ((bi - ai @ xi) ** 2).mean() <= var, i
