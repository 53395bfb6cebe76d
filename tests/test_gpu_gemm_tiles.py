"""Every tile the GEMM chooses (gemm.hip: 128, 64 and 32, K whole or split over
groups of wavefronts) at ragged sizes, K shorter than a slab and K that leaves
groups without a slab.  Entries are small integers, so every product and sum is
exact in both types and the result has to equal the integer one bit for bit
(Matrix::mul, src/matrix/mod.rs:957-980)."""
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (33, 31, 65), (64, 64, 192), (257, 255, 191), (500, 500, 1023),   # 32
          (65, 40, 2100), (700, 1100, 70), (1000, 777, 300), (1300, 1025, 257),        # 64, K split
          (1600, 1500, 33), (2100, 2047, 18),                                          # 64
          (4097, 4100, 17), (4223, 4100, 40)]                                          # 128


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("name", ["f64", "f32"])
def test_integer_products(tctx, torch_cuda, m, n, k, name):
    torch = torch_cuda
    dt = torch.float64 if name == "f64" else torch.float32
    g = torch.Generator(device="cuda").manual_seed(m + n + k)

    def ints(r, c, pad):        # rows of a wider matrix; NaN where nothing may be used
        t = torch.full((r, c + pad), float("nan"), dtype=dt, device="cuda")
        t[:, :c] = torch.randint(-3, 4, (r, c), generator=g, device="cuda").to(dt)
        return t
    A, B, C = ints(m, k, 3), ints(k, n, 5), ints(m, n, 1)
    want = C[:, :n].cpu().double() * 2.0 - A[:, :k].cpu().double() @ B[:, :n].cpu().double()
    (tctx.gemm_dev if name == "f64" else tctx.sgemm_dev)(A[:, :k], B[:, :n], C[:, :n], -1.0, 2.0)
    torch.cuda.synchronize()
    assert torch.equal(C[:, :n].cpu().double(), want)
    assert torch.isnan(C[:, n:]).all()
