"""What follows a bounded wait that is given up inside the LU: LA_ERR_TIMEOUT,
no row moved by a swap list that was never written, and a context that goes
on.  A limit of 0 ms (LAHIP_SPIN_LIMIT_MS) makes the waits give up at once;
every kernel still ends normally.  The larger factorisation before it leaves
swap lists with rows the smaller matrix does not have."""
import pytest

import la_hip

pytestmark = pytest.mark.gpu


def _factor(ctx, torch, W):
    piv = torch.empty(W.shape[0], dtype=torch.int64, device="cuda")
    info = torch.full((4,), -7, dtype=torch.int32, device="cuda")
    ctx.getrf_dev(W, piv, info)
    torch.cuda.synchronize()
    return piv, info


# the column-distributed block, with and without look-ahead, and the
# row-distributed panel (more rows than the block's tallest layout)
@pytest.mark.parametrize("shape,lookahead", [((600, 600), "1"), ((600, 600), "0"),
                                             ((8300, 128), "0")])
def test_given_up_wait(tctx, torch_cuda, monkeypatch, shape, lookahead):
    torch = torch_cuda
    m, n = shape
    print(f"given-up wait {shape} look-ahead {lookahead}", flush=True)
    monkeypatch.setenv("LAHIP_LOOKAHEAD", lookahead)
    big = torch.randn(m + 2000, n + 100, dtype=torch.float64, device="cuda")
    _factor(tctx, torch, big)
    A = torch.randn(m, n, dtype=torch.float64, device="cuda")
    ref = A.clone()
    p0, i0 = _factor(tctx, torch, ref)
    assert i0[1].item() == la_hip.LA_OK
    frame = torch.full((m + 512, n + 64), 7.0, dtype=torch.float64, device="cuda")
    W = frame[256:256 + m, 32:32 + n]
    W.copy_(A)
    monkeypatch.setenv("LAHIP_SPIN_LIMIT_MS", "0")
    piv, info = _factor(tctx, torch, W)
    monkeypatch.delenv("LAHIP_SPIN_LIMIT_MS")
    assert info[1].item() == la_hip.LA_ERR_TIMEOUT
    assert torch.equal(piv.sort().values.cpu(), torch.arange(m))
    W.fill_(7.0)
    assert (frame == 7.0).all()
    p1, i1 = _factor(tctx, torch, A)
    assert torch.equal(p0, p1) and torch.equal(ref, A) and torch.equal(i0[:2], i1[:2])
