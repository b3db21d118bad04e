"""float32 GELU over its whole range, as the epilogue of a product that is zero (so that its input is the bias alone): around zero, about the
end of the polynomial's range, far out on both sides.

Bound: three half-ulps of 1 times |x| (exponential, G and the last product; the fit is off by 7e-9)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

import test_gpu_f32_split as f32  # noqa: E402
from test_gpu_f32_split import lib as lib  # noqa: E402,F401


@pytest.mark.parametrize("tile", [128, 95, 103])
def test_gelu_of_every_magnitude(lib, tile):  # noqa: F811
    mags = np.concatenate([[0.0], 2.0 ** np.arange(-40, 100, 3.0), np.linspace(0.01, 6.5, 650), [5.0, np.nextafter(np.float32(5), np.float32(6))]])
    x = np.concatenate([mags, -mags]).astype(np.float32)
    x = np.pad(x, (0, -len(x) % 32))
    N, K = len(x), 64
    X, W = f32.split(lib, torch.zeros(1, K, device="cuda")), f32.split(lib, torch.randn(N, K, device="cuda"))
    b = torch.from_numpy(x).cuda()
    Y = torch.zeros(lib.cubert_split_bytes(1, N), dtype=torch.uint8, device="cuda")
    f32.check(lib.cubert_op_gemm(X.data_ptr(), W.data_ptr(), b.data_ptr(), Y.data_ptr(), 1, N, K, K, f32.SPLIT, f32.SPLIT, 1, tile, 0, None))
    torch.cuda.synchronize()
    z = torch.from_numpy(x).double()
    want = 0.5 * z * torch.special.erfc(-z / np.sqrt(2.0))
    err = (f32.unsplit(Y, 1, N)[0].cpu() - want).abs()
    assert (err <= 3 * 2.0 ** -24 * z.abs()).all()


@pytest.mark.parametrize("tile", [128, 95, 103])
def test_gelu_interval_by_interval(lib, tile):  # noqa: F811
    """Both sides of zero and of the point where the two forms meet.  Bound, u = 2^-24.  Below 1: x^2 R rounds at x^2, at R (an ulp of 0.4 and what the
    products before it leave, together 1.1 u) and at the end.  From 1 on, t = a e P: the exponential is off by an ulp and by its argument's two roundings
    (x^2 u), P by 3 u where its terms cancel least (next to 1), the product by u, and the fit by 4.6e-9; the end rounds once."""
    x = np.concatenate([np.random.default_rng(1).uniform(lo, hi, 1500) for lo, hi in
                        [(0, 0.25), (0.25, 0.5), (0.5, 0.75), (0.75, 0.99), (0.99, 1.01), (1.01, 1.5), (1.5, 2), (2, 3), (3, 4), (4, 5), (5, 6), (6, 9)]])
    x = np.concatenate([x, -x]).astype(np.float32)
    N, K = len(x), 64
    X, W = f32.split(lib, torch.zeros(1, K, device="cuda")), f32.split(lib, torch.randn(N, K, device="cuda"))
    b = torch.from_numpy(x).cuda()
    Y = torch.zeros(lib.cubert_split_bytes(1, N), dtype=torch.uint8, device="cuda")
    f32.check(lib.cubert_op_gemm(X.data_ptr(), W.data_ptr(), b.data_ptr(), Y.data_ptr(), 1, N, K, K, f32.SPLIT, f32.SPLIT, 1, tile, 0, None))
    torch.cuda.synchronize()
    z = torch.from_numpy(x).double()
    want = 0.5 * z * torch.special.erfc(-z / np.sqrt(2.0))
    err = (f32.unsplit(Y, 1, N)[0].cpu() - want).abs()
    u, tail = 2.0 ** -24, 0.5 * z.abs() * torch.special.erfc(z.abs() / np.sqrt(2.0))
    bound = torch.where(z.abs() < 1, u * (want.abs() + 1.5 * z * z) + 4e-10, u * (want.abs() + (6 + z * z) * tail) + 4.6e-9)
    assert (err <= bound).all(), (x[(err > bound).numpy()][:5], float((err / bound).max()))
