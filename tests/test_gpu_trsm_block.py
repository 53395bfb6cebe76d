"""LU solves with several right-hand sides (trsm_block.hip and one GEMM per 256
rows) at the edges of their blocks: 64-row panels, 256-row blocks, sixteen
columns per workgroup; against LUDecomposition::solve (src/decomp/lu.rs:237-278)
and the inverse (src/matrix/mod.rs:1034-1037)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


@pytest.mark.parametrize("n", [65, 127, 192, 255, 256, 257, 321, 511, 513, 770])
@pytest.mark.parametrize("nrhs", [1, 2, 15, 16, 17, 33])
def test_few_columns(ctx, n, nrhs):
    a, b = oracle.uniform(5, n, (n, n)), oracle.uniform(6, nrhs, (n, nrhs))
    lu, piv, _ = ctx.lu_new(a)
    x = ctx.lu_solve(lu, piv, b)
    ref = oracle.lu_solve(lu, piv, b)
    # both solve the same factor: forward error of a triangular pair, n u cond each
    tol = 2 * n * U * np.linalg.cond(a, np.inf)
    assert np.abs(x - ref).max() <= tol * np.abs(ref).max()


# Triangles of small integers with unit diagonals: no step rounds, so the
# solution equals the integer one bit for bit
@pytest.mark.parametrize("n", [65, 200, 300])
def test_integer_triangles(ctx, n):
    rng = np.random.default_rng(n)
    low = np.eye(n) + np.diag(rng.integers(-1, 2, size=n - 1), -1)
    up = np.eye(n) + np.diag(rng.integers(-1, 2, size=n - 1), 1)
    xs = rng.integers(-4, 5, size=(n, 3)).astype(float)
    lu = np.tril(low, -1) + up
    x = ctx.lu_solve(lu, np.arange(n, dtype=np.uint64), low @ (up @ xs))
    assert np.array_equal(x, xs)


# Upper triangles of factors with singular values in [1e-6, 1] (L the identity):
# after the correction x carries its own rounding (at most u, rms u / 3^(1/2))
# and that of the residual, a sum of at most 100 terms whose rounding is below
# a tenth of u of the sum of their magnitudes: 0.58 + 0.07 u.
@pytest.mark.parametrize("n", [65, 100])
def test_small_solve_residual(tctx, torch_cuda, n):
    torch = torch_cuda
    rng = np.random.default_rng(n)
    total = []
    for k in range(12):
        q1, q2 = (np.linalg.qr(rng.standard_normal((n, n)))[0] for _ in range(2))
        lu = torch.linalg.lu_factor(torch.from_numpy((q1 * 1e-6 ** np.linspace(0, 1, n)) @ q2))[0]
        W, B = torch.triu(lu).cuda(), torch.randn(n, 16, dtype=torch.float64, device="cuda")
        X, piv = torch.empty_like(B), torch.arange(n, device="cuda")
        tctx.getrs_dev(W, piv, B, X)
        torch.cuda.synchronize()
        u, x, b = (t.cpu().numpy().astype(np.longdouble) for t in (W, X, B))
        total.append(((b - u @ x) / (np.abs(u) @ np.abs(x))) ** 2)
    assert np.mean(total) ** 0.5 <= 0.65 * 2.0 ** -53
