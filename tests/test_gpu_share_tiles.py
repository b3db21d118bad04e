"""GEMM tiles on split operands whose four waves share K (32, 64 and 96 features x 128 tokens): K steps that the waves of all parts do not
share evenly, waves with a single step, odd and even counts of them, rows and features that end inside a tile, a tile grid that the XCDs do
not divide evenly; every epilogue.

Bounds as in the test of the split layout: 6 K / 16 float32 accumulations a result and a few additions (partial sums of four waves, parts, bias,
residual) against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

import test_gpu_f32_split as f32  # noqa: E402
from test_gpu_f32_split import lib as lib  # noqa: E402,F401

TILES = (101, 102, 103)
U = 2.0 ** -24


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K,splits", [(1, 4, 64, 1), (33, 100, 80, 1), (129, 96, 192, 3), (300, 196, 1040, 2), (1025, 264, 512, 5), (257, 1160, 336, 1)])
def test_float32_result_in_parts(lib, tile, M, N, K, splits):  # noqa: F811
    X, W, b = f32.operands(M, N, K)
    R = torch.randn(M, N, generator=torch.Generator().manual_seed(2))
    want = X.double() @ W.double().t() + b.double() + R.double()
    scale = X.double().abs() @ W.double().abs().t() + b.double().abs() + R.double().abs()
    xs, ws, bd, Rd = f32.split(lib, X.cuda()), f32.split(lib, W.cuda()), b.cuda(), R.cuda()
    Y = torch.full((splits + 1, M, N), float("nan"), device="cuda")
    f32.check(lib.cubert_op_gemm_residual(xs.data_ptr(), ws.data_ptr(), bd.data_ptr(), Rd.data_ptr(), Y.data_ptr(), M, N, K, K, f32.SPLIT, tile,
                                          splits << 8 if splits > 1 else 0, None))
    torch.cuda.synchronize()
    assert torch.isnan(Y[splits]).all()                  # nothing past the last part
    assert ((Y[:splits].double().sum(0).cpu() - want).abs() <= (6 * K / 16 + 6 + splits) * U * scale).all()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K", [(1, 32, 64), (70, 160, 144), (257, 288, 96)])
def test_gelu_result(lib, tile, M, N, K):  # noqa: F811
    X, W, b = f32.operands(M, N, K)
    z = X.double() @ W.double().t() + b.double()
    scale = X.double().abs() @ W.double().abs().t() + b.double().abs()
    xs, ws, bd = f32.split(lib, X.cuda()), f32.split(lib, W.cuda()), b.cuda()
    Y = torch.full((lib.cubert_split_bytes(M, N) + 4096,), 0x55, dtype=torch.uint8, device="cuda")
    f32.check(lib.cubert_op_gemm(xs.data_ptr(), ws.data_ptr(), bd.data_ptr(), Y.data_ptr(), M, N, K, K, f32.SPLIT, f32.SPLIT, 1, tile, 0, None))
    torch.cuda.synchronize()
    assert (Y[-4096:] == 0x55).all()
    err = (f32.unsplit(Y[:-4096], M, N).cpu() - 0.5 * z * (1 + torch.erf(z / np.sqrt(2.0)))).abs()
    # |gelu'| < 1.13; the function and the products in it add a few roundings of |z|
    assert (err <= 1.13 * (6 * K / 16 + 6) * U * scale + 8 * U * z.abs()).all()


@pytest.mark.parametrize("B,S,heads,tile", [(1, 1, 1, 101), (3, 45, 2, 101), (2, 33, 2, 102), (2, 129, 3, 103), (1, 300, 1, 103)])
def test_qkv_and_attention(lib, B, S, heads, tile):  # noqa: F811
    f32.test_qkv_projection_and_attention(lib, B, S, heads, tile)


def test_refused(lib):  # noqa: F811
    """A wave without a K step, operands of another kind."""
    d = torch.zeros(1 << 16, dtype=torch.uint8, device="cuda")
    p = d.data_ptr()
    assert lib.cubert_op_gemm(p, p, p, p, 32, 32, 48, 48, f32.SPLIT, 0, 0, 103, 0, None) != 0
    assert lib.cubert_op_gemm_residual(p, p, p, p, p, 32, 32, 64, 64, f32.SPLIT, 103, 2 << 8, None) != 0
    assert lib.cubert_op_gemm(p, p, p, p, 32, 32, 64, 64, 1, 0, 0, 103, 3, None) != 0
    assert lib.cubert_op_gemm(p, p, p, p, 32, 32, 64, 64, 0, 0, 0, 103, 0, None) != 0
