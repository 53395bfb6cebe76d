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
