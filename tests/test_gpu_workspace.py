"""The dense solvers under a workspace limit, inside a capture and on a stream
of few CUs: the paths taken where the optional buffers have no room, and what
the limits hold.  Each test has a context of its own, whose workspaces start
empty.  Results are compared with the unlimited context's (the same
factorisation with other roundings) or with numpy."""
import ctypes

import numpy as np
import pytest

import la_hip

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.fixture
def fresh(torch_cuda):
    """A context on a side stream of its own, as captures need."""
    stream = torch_cuda.cuda.Stream()
    c = la_hip.Context(0)
    c.set_stream(stream.cuda_stream)
    c.side = stream
    yield c
    torch_cuda.cuda.synchronize()
    c.close()


def _limit(ctx, nbytes):
    assert ctx.lib.la_ctx_set_workspace_limit(ctx.h, nbytes) == 0


def _lu(ctx, torch, A):
    W = A.clone()
    piv = torch.empty(A.shape[0], dtype=torch.int64, device="cuda")
    info = torch.zeros(4, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    ctx.getrf_dev(W, piv, info)
    torch.cuda.synchronize()
    assert info[1].item() == la_hip.LA_OK
    return W, piv


def _backward_stable(torch, A, W, piv):
    """|PA - LU| <= n u |L||U|, twice that for the product formed here."""
    k = min(A.shape)
    L = torch.tril(W[:, :k], -1) + torch.eye(A.shape[0], k, dtype=W.dtype, device="cuda")
    U = torch.triu(W[:k])
    bound = 2 * k * 2.0 ** -53 * (L.abs() @ U.abs())
    return ((A[piv] - L @ U).abs() <= bound).all().item()


# 8 MiB hold the row-distributed panels' workspace and not the block kernel's
# slot (16 MiB).
@pytest.mark.parametrize("shape", [(600, 600), (2049, 2049), (300, 700), (3000, 190)])
def test_lu_without_block_slot(fresh, tctx, torch_cuda, shape):
    torch = torch_cuda
    A = torch.randn(shape, dtype=torch.float64, device="cuda")
    W0, p0 = _lu(tctx, torch, A)
    _limit(fresh, 8 * MIB)
    W1, p1 = _lu(fresh, torch, A)
    assert torch.equal(p0, p1) and _backward_stable(torch, A, W1, p1)
    _limit(fresh, 0)
    W2, p2 = _lu(fresh, torch, A)
    assert torch.equal(p0, p2) and torch.equal(W0, W2)


# What la_dgetrf_dev took before the block kernel had a slot: panel workspace
# (and, with more than one block, the look-ahead's second set) and swap list.
@pytest.mark.parametrize("n,limit", [(200, 671744 + 4096), (300, 819200 + 4096)])
def test_lu_least_limit(fresh, torch_cuda, n, limit):
    A = torch_cuda.randn(n, n, dtype=torch_cuda.float64, device="cuda")
    _limit(fresh, limit)
    _lu(fresh, torch_cuda, A)


# A later slot takes the block kernel's room; the next LU goes without.
def test_block_slot_makes_room(fresh, tctx, torch_cuda):
    torch = torch_cuda
    A = torch.randn(900, 900, dtype=torch.float64, device="cuda")
    W0, p0 = _lu(tctx, torch, A)
    _limit(fresh, 20 * MIB)
    W1, p1 = _lu(fresh, torch, A)
    assert torch.equal(W0, W1)
    a, b = np.random.default_rng(0).standard_normal((2, 700, 700))
    assert np.abs(fresh.mul(a, b) - a @ b).max() <= 1e-11     # 11.8 MiB of host buffers
    W2, p2 = _lu(fresh, torch, A)
    assert torch.equal(p0, p2) and _backward_stable(torch, A, W2, p2)


# Solves: 64-row exchange (limit) and 256-row blocks, from either side of
# their rule (n = 64 | 65, 512 | 513 with one right-hand side).
@pytest.mark.parametrize("n", [64, 65, 256, 257, 512, 513, 1000])
@pytest.mark.parametrize("limit", [0, 4 * MIB])
def test_solve_paths(fresh, torch_cuda, n, limit):
    torch = torch_cuda
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 2 * np.sqrt(n) * np.eye(n)
    W, piv = _lu(fresh, torch, torch.from_numpy(a).cuda())
    fresh2 = la_hip.Context(0)
    fresh2.set_stream(fresh.side.cuda_stream)
    _limit(fresh2, limit)
    for nrhs in (1, 2, 7, 16, 17):
        b = rng.standard_normal((n, nrhs))
        B = torch.from_numpy(b).cuda()
        X = torch.empty_like(B)
        torch.cuda.synchronize()
        fresh2.getrs_dev(W, piv, B, X)
        torch.cuda.synchronize()
        x = X.cpu().numpy()
        # backward stable solves: residual within 3 n u |L||U||x|, growth < 2 here
        r = np.abs(b - a @ x).max(0)
        assert (r <= 6 * n * 2.0 ** -53 * np.abs(a).sum(1).max() * np.abs(x).max(0)).all(), nrhs
    fresh2.close()


@pytest.mark.parametrize("limit", [0, 3 * MIB])
def test_qr_small_pool(fresh, torch_cuda, limit):
    torch = torch_cuda
    rng = np.random.default_rng(5)
    a, b = rng.standard_normal((700, 300)), rng.standard_normal((700, 3))
    W, rd = torch.from_numpy(a).cuda(), torch.empty(300, dtype=torch.float64, device="cuda")
    B, X = torch.from_numpy(b).cuda(), torch.empty(300, 3, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    _limit(fresh, limit)
    fresh.geqrf_dev(W, rd)
    assert fresh.qrs_dev(W, rd, B, X) == la_hip.LA_OK
    torch.cuda.synchronize()
    want = np.linalg.lstsq(a, b, rcond=None)[0]
    # kappa(a) < 6: m n^(1/2) u kappa^2 and the reference's own error
    assert np.abs(X.cpu().numpy() - want).max() <= 700 * 18 * 2.0 ** -53 * 36


# A captured factorisation and solve (the plain schedule, whatever its size),
# replayed on other data.  The context is warm, as captures need; `limit`:
# between capture and replay another slot asks for room, which the captured
# block slot must not give.
@pytest.mark.parametrize("n", [200, 700])
@pytest.mark.parametrize("limit", [False, True])
def test_captured_lu_solve(fresh, tctx, torch_cuda, n, limit):
    torch = torch_cuda
    A = torch.randn(n, n, dtype=torch.float64, device="cuda")
    B = torch.randn(n, 4, dtype=torch.float64, device="cuda")
    W, X = torch.empty_like(A), torch.empty_like(B)
    piv = torch.empty(n, dtype=torch.int64, device="cuda")
    info = torch.zeros(4, dtype=torch.int32, device="cuda")

    def call():
        W.copy_(A)
        fresh.getrf_dev(W, piv, info)
        fresh.getrs_dev(W, piv, B, X)

    torch.cuda.synchronize()
    with torch.cuda.stream(fresh.side):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=fresh.side):
        call()
    for k in range(3):
        if limit:
            _limit(fresh, 20 * MIB)
            a = np.ones((700, 700))
            with pytest.raises(la_hip.LaError) as e:
                fresh.mul(a, a)                 # 11.8 MiB beside the 16 that stay
            assert e.value.status == la_hip.LA_ERR_NOMEM
        A.normal_()
        B.normal_()
        W0, p0 = _lu(tctx, torch, A)
        X0 = torch.empty_like(B)
        tctx.getrs_dev(W0, p0, B, X0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(W, W0) and torch.equal(piv, p0) and torch.equal(X, X0), k


# A solve captured where the inverses' buffer would have to grow: the 64-row
# exchange takes it.
def test_captured_solve_without_room(fresh, torch_cuda):
    torch, n = torch_cuda, 700
    a = np.random.default_rng(2).standard_normal((n, n)) + 50 * np.eye(n)
    W, piv = _lu(fresh, torch, torch.from_numpy(a).cuda())
    B = torch.randn(n, 4, dtype=torch.float64, device="cuda")
    X, b1, x1 = torch.empty_like(B), B[:, :1].contiguous(), torch.empty_like(B[:, :1])
    torch.cuda.synchronize()
    fresh.getrs_dev(W, piv, b1, x1)             # one column: the exchange's buffer
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=fresh.side):
        fresh.getrs_dev(W, piv, B, X)
    graph.replay()
    torch.cuda.synchronize()
    want = np.linalg.solve(a, B.cpu().numpy())
    assert np.abs(X.cpu().numpy() - want).max() <= 1e-12 * np.abs(want).max()


# A caller's stream with one CU of each XCD: a block of 16 workgroups goes to
# the row-distributed panel (8 of 128 rows), one of 8 stays.
@pytest.mark.parametrize("shape", [(900, 200), (500, 200)])
def test_stream_of_few_cus(tctx, torch_cuda, shape):
    torch = torch_cuda
    hip = tctx.lib                              # its HIP runtime's symbols with it
    s, words = ctypes.c_void_p(), (ctypes.c_uint32 * 8)(0xff)
    assert hip.hipExtStreamCreateWithCUMask(ctypes.byref(s), 8, words) == 0
    c = la_hip.Context(0)
    c.set_stream(s.value)
    A = torch.randn(shape, dtype=torch.float64, device="cuda")
    W0, p0 = _lu(tctx, torch, A)
    W1, p1 = _lu(c, torch, A)
    assert torch.equal(p0, p1) and _backward_stable(torch, A, W1, p1)
    c.close()
    assert hip.hipStreamDestroy(s) == 0
