"""The skinny tiles at row counts at which a tile's number times the rows' tiles, or a token times the line's length, passes 2^32: the last tile of every
band, and the last position of the later lines, of a product and of Q, K, V.

Bound as at their other sizes: K / 16 float32 accumulations and a few additions of bf16 products; the reference here is a float32 product, which adds
K accumulations of its own."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from test_gpu_units_layout import UNITS, check  # noqa: E402
from test_gpu_units_layout import lib as lib  # noqa: E402,F401

U = 2.0 ** -24


def pack(rows):
    """[R, K] bf16 on the GPU in the units layout (R a multiple of 32; blocks of 256 rows)."""
    R, K = rows.shape
    full = torch.zeros((R + 255) // 256 * 256, K, dtype=torch.bfloat16, device="cuda")
    full[:R] = rows
    return full.view(-1, 8, 32, K // 32, 2, 2, 8).permute(0, 3, 1, 4, 5, 2, 6).contiguous()


def operands(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(7)
    X = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    W = (torch.randn(N, K, generator=g, device="cuda") * 0.05).to(torch.bfloat16)
    return X, W, torch.randn(N, generator=g, device="cuda")


def within(got, X, W, b, extra=0.0):
    """Row blocks of a result against a float32 product."""
    K = X.shape[1]
    for r in range(0, len(X), 1 << 18):
        x = X[r:r + (1 << 18)].float()
        want, scale = x @ W.float().t() + b, x.abs() @ W.float().abs().t() + b.abs()
        err = (got[r:r + (1 << 18)].float() - want).abs()
        assert bool((err <= (K / 16 + K + 8) * U * scale + extra * want.abs()).all()), r


def test_rows_tiles_past_32_bits(lib):  # noqa: F811
    M, N, K = 32 * 37927, 128, 128                               # 37927: 2^32 divided by it leaves little, the third band ends past it
    X, W, b = operands(M, N, K)
    guard = 64                                                   # rows in front of the result and behind it
    Y = torch.full((M + 2 * guard, N), float("nan"), device="cuda")
    xp, wp = pack(X), pack(W)
    check(lib.cubert_op_gemm(xp.data_ptr(), wp.data_ptr(), b.data_ptr(), Y[guard:].data_ptr(), M, N, K, K, 1, 0, 0, 95, 3 | UNITS["X"] | UNITS["W"], None))
    torch.cuda.synchronize()
    assert bool(torch.isnan(Y[:guard]).all()) and bool(torch.isnan(Y[guard + M:]).all())
    within(Y[guard:guard + M], X, W, b)


def test_positions_past_32_bits(lib):  # noqa: F811
    B, S, H = 260, 4096, 128
    X, W, b = operands(B * S, 3 * H, H)
    xp, wp = pack(X), pack(W)
    out = torch.zeros(3, B * S, H, dtype=torch.bfloat16, device="cuda")
    check(lib.cubert_op_gemm_qkv(xp.data_ptr(), wp.data_ptr(), b.data_ptr(), *[t.data_ptr() for t in out], B, S, 2, 1, 97, 3 | UNITS["X"] | UNITS["W"] | 32, None))
    torch.cuda.synchronize()
    for i in range(3):
        within(out[i].view(B, 2, S, 64).transpose(1, 2).reshape(B * S, H), X, W[i * H:(i + 1) * H], b[i * H:(i + 1) * H], 2.0 ** -8)
