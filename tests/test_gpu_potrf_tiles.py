"""Dense Cholesky (potrf.hip) at the edges of its 16 x 16 tiles, 64-column
panels and 256-column blocks, and through the branch its tiles take for
non-finite values and pivots outside the fast square root's range
(CholeskyDecomposition::new, src/decomp/cholesky.rs:56-110)."""
import numpy as np
import pytest

import la_hip
import oracle

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def _factor(tctx, torch, a):
    W = torch.from_numpy(a).cuda()
    st = torch.zeros(1, dtype=torch.int32, device="cuda")
    tctx.potrf_dev(W, st)
    torch.cuda.synchronize()
    return W.cpu().numpy(), int(st.item())


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 48, 63, 64, 65, 79, 81, 127, 129, 255,
                               257, 300, 320])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -600, 2.0 ** 600])
def test_backward_error(tctx, torch_cuda, n, scale):
    g = oracle.uniform(9, n, (n, n))
    a = g @ g.T
    a = (a + a.T) * 0.5 + np.eye(n)
    l, st = _factor(tctx, torch_cuda, a * scale)
    assert st == la_hip.LA_OK and np.array_equal(l, np.tril(l))
    # |A - L L^T| <= (n + 1) u |L||L^T| elementwise; the second term is the
    # rounding of the check itself.  Powers of four scale L exactly.
    l = l / np.sqrt(scale)
    assert (np.abs(a - l @ l.T) <= 2 * (n + 2) * U * (np.abs(l) @ np.abs(l.T))).all()


@pytest.mark.parametrize("n,k,v", [(70, 0, np.nan), (70, 20, np.nan), (70, 69, np.nan),
                                   (70, 20, -1.0), (70, 20, 0.0), (100, 66, -1.0),
                                   (70, 40, np.inf)])
def test_bad_pivots(tctx, torch_cuda, n, k, v):
    a = np.eye(n) * 4.0
    a[n - 1, :] = a[:, n - 1] = 1.0
    a[n - 1, n - 1] = 400.0
    a[k, k] = v
    l, st = _factor(tctx, torch_cuda, a)
    ref, _ = oracle.chol_new(a)
    assert st == (la_hip.LA_OK if ref is not None else la_hip.LA_NOT_SPD)
    if ref is not None:
        assert np.array_equal(np.isnan(l), np.isnan(ref))
        assert np.allclose(np.nan_to_num(l), np.nan_to_num(ref), rtol=1e-14, atol=0)


# the batched kernel (batched_chol.hip): the same bound for its factors, and for
# its solutions the backward error of two triangular solves with them
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -600, 2.0 ** 600])
def test_batched_backward_error(tctx, torch_cuda, scale):
    torch = torch_cuda
    sizes = np.array([1, 7, 8, 9, 15, 16, 17, 24, 25, 33, 64, 65, 128, 129, 255, 256])
    offA = np.concatenate([[0], np.cumsum(sizes ** 2)[:-1]])
    offB = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    mats, rhs = [], []
    for n in sizes:
        g = oracle.uniform(9, n, (n, n))
        a = g @ g.T
        mats.append((a + a.T) * 0.5 + np.eye(n))
        rhs.append(oracle.uniform(10, n, (n,)))
    A = torch.from_numpy(np.concatenate([m.ravel() for m in mats]) * scale).cuda()
    B = torch.from_numpy(np.concatenate(rhs)).cuda()
    L, X = torch.full_like(A, float("nan")), torch.full_like(B, float("nan"))
    st = torch.full((len(sizes),), -1, dtype=torch.int32, device="cuda")
    dA, dB = torch.from_numpy(offA).cuda(), torch.from_numpy(offB).cuda()
    plan = tctx.batch_plan(0, sizes)
    tctx.potrf_potrs_batched_dev(plan, dA, dB, A, L, B, X, st)
    torch.cuda.synchronize()
    plan.close()
    assert (st.cpu().numpy() == 0).all()
    lh, xh = L.cpu().numpy() / np.sqrt(scale), X.cpu().numpy() * scale
    for n, oa, ob, a, b in zip(sizes, offA, offB, mats, rhs):
        l, x = lh[oa:oa + n * n].reshape(n, n), xh[ob:ob + n]
        assert np.array_equal(l, np.tril(l))
        ll = np.abs(l) @ np.abs(l.T)
        assert (np.abs(a - l @ l.T) <= 2 * (n + 2) * U * ll).all()
        assert (np.abs(b - a @ x) <= 4 * (n + 2) * U * (ll @ np.abs(x) + np.abs(b))).all()
