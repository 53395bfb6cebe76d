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
