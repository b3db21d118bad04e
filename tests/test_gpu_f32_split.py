"""float32 mode's kernels on operands split into three bf16 planes, against float64: the GEMM tiles at the edges of their
tiles, K shares and row blocks, and the attention at the edges of its key and query blocks.

Bounds.  An element is the exact sum of its planes; of the nine plane products of a pair the six that are formed miss the
float32 product by less than 2^-24 of it.  The 6 K / 16 accumulations of an output round once each in float32, so its error
stays below (6 K / 16 + 2) 2^-24 sum |x w| (worst case), and its root mean square over many outputs near
sqrt(6 K / 16) 2^-24 of the result's; a plane left out anywhere (2^-18 and more) would break the latter."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
SPLIT, U = 2, 2.0 ** -24
SKINNY12, SKINNY22, T256x128 = 97, 98, 384


@pytest.fixture(scope="module")
def lib():
    from cudabert_amd import pybert
    lib = pybert.lib
    lib.cubert_split_bytes.argtypes = [ctypes.c_size_t] * 2
    lib.cubert_split_bytes.restype = ctypes.c_size_t
    lib.cubert_op_split_operand.argtypes = [ctypes.c_void_p] * 2 + [ctypes.c_int] * 3 + [ctypes.c_void_p]
    return lib


def check(rc):
    from cudabert_amd import pybert
    pybert.check(rc)


def split(lib, a):
    R, K = a.shape
    d = torch.zeros(lib.cubert_split_bytes(R, K), dtype=torch.uint8, device="cuda")
    t = a.t().contiguous()
    check(lib.cubert_op_split_operand(t.data_ptr(), d.data_ptr(), K, R, 0, None))
    torch.cuda.synchronize()
    return d


def unsplit(d, R, K):
    """[rows, K] float64 from the split layout: units [row / 32, k / 16, plane], lane 32 (k / 8 % 2) + row % 32."""
    u = d.view(torch.bfloat16).view(-1, K // 16, 3, 2, 32, 8)[: (R + 31) // 32].double()
    return u.sum(2).permute(0, 3, 1, 2, 4).reshape(-1, K)[:R]


def operands(M, N, K, seed=5):
    g = torch.Generator().manual_seed(seed)
    X = torch.randn(M, K, generator=g) * torch.exp2(torch.randint(-6, 7, (M, 1), generator=g).float())
    W = torch.randn(N, K, generator=g) * 0.05
    return X, W, torch.randn(N, generator=g)


def assert_close(got, want, scale, K):
    err = (got - want).abs()
    steps = 6 * K / 16
    assert (err <= (steps + 2) * U * scale).all(), float((err / scale).max() / U)
    assert float(err.norm() / want.norm()) < np.sqrt(steps) * U


def test_split_planes_hold_the_number_exactly(lib):
    g = torch.Generator().manual_seed(1)
    a = torch.randn(40, 48, generator=g) * torch.exp2(torch.randint(-60, 61, (40, 48), generator=g).float())
    assert torch.equal(unsplit(split(lib, a.cuda()), 40, 48).cpu(), a.double())


@pytest.mark.parametrize("tile", [128, T256x128, SKINNY12, SKINNY22])
@pytest.mark.parametrize("M,N,K,splits", [(1, 32, 64, 1), (33, 128, 64, 1), (127, 96, 80, 1), (130, 264, 256, 2), (65, 520, 512, 4)])
def test_gemm(lib, tile, M, N, K, splits):
    X, W, b = operands(M, N, K)
    R = torch.randn(M, N, generator=torch.Generator().manual_seed(9))
    want = X.double() @ W.double().t() + b.double() + R.double()
    scale = X.double().abs() @ W.double().abs().t() + b.double().abs() + R.double().abs()
    xs, ws, bd, Rd = split(lib, X.cuda()), split(lib, W.cuda()), b.cuda(), R.cuda()
    Y = torch.full((splits + 1, M, N), float("nan"), device="cuda")
    flags = (splits << 8) if splits > 1 else 0
    check(lib.cubert_op_gemm_residual(xs.data_ptr(), ws.data_ptr(), bd.data_ptr(), Rd.data_ptr(), Y.data_ptr(), M, N, K, K, SPLIT,
                                      tile, flags, None))
    torch.cuda.synchronize()
    assert torch.isnan(Y[splits]).all()                  # nothing past the last part
    assert_close(Y[:splits].double().sum(0).cpu(), want, scale, K)


@pytest.mark.parametrize("tile", [128, T256x128, SKINNY12, SKINNY22])
@pytest.mark.parametrize("M,N,K", [(1, 32, 64), (70, 160, 128), (257, 288, 96)])
def test_gelu_result_is_the_next_split_operand(lib, tile, M, N, K):
    X, W, b = operands(M, N, K)
    z = X.double() @ W.double().t() + b.double()
    scale = X.double().abs() @ W.double().abs().t() + b.double().abs()
    xs, ws, bd = split(lib, X.cuda()), split(lib, W.cuda()), b.cuda()
    Y = torch.zeros(lib.cubert_split_bytes(M, N), dtype=torch.uint8, device="cuda")
    check(lib.cubert_op_gemm(xs.data_ptr(), ws.data_ptr(), bd.data_ptr(), Y.data_ptr(), M, N, K, K, SPLIT, SPLIT, 1, tile, 0, None))
    torch.cuda.synchronize()
    err = (unsplit(Y, M, N).cpu() - 0.5 * z * (1 + torch.erf(z / np.sqrt(2.0)))).abs()
    # |gelu'| < 1.13; erff and the products after it add a few roundings of |z|
    assert (err <= 1.13 * (6 * K / 16 + 2) * U * scale + 8 * U * z.abs()).all()


@pytest.mark.parametrize("B,S,heads,tile", [(1, 1, 1, 0), (2, 33, 2, 128), (3, 64, 2, T256x128), (2, 129, 3, SKINNY12),
                                            (1, 200, 2, SKINNY22), (2, 300, 1, 128), (1, 545, 1, SKINNY12)])
def test_qkv_projection_and_attention(lib, B, S, heads, tile):
    H, Sp = heads * 64, (S + 31) // 32 * 32
    X, W, b = operands(B * S, 3 * H, H)
    X = X / X.abs().max() * 4
    qkv = (X.double() @ W.double().t() * 4 + b.double()).view(B, S, 3, heads, 64).permute(2, 0, 3, 1, 4)
    W = W * 4
    scale_in = float((X.double().abs() @ W.double().abs().t() + b.double().abs()).max())
    rng = np.random.default_rng(3)
    mask = np.zeros((B, Sp), np.float32)
    mask[:, S:] = -np.inf
    for i in range(B):
        n = int(rng.integers(1, S + 1)) if i else S
        mask[i, n:S] = -10000.0
    m = torch.from_numpy(mask)
    sc = torch.matmul(qkv[0], qkv[1].transpose(-1, -2).contiguous()) * 0.125 + m[:, None, None, :S].double()
    want = torch.matmul(torch.softmax(sc, -1), qkv[2]).permute(0, 2, 1, 3).reshape(B * S, H)
    xs, ws, bd, md = split(lib, X.cuda()), split(lib, W.cuda()), b.cuda(), m.cuda()
    q, k, v = (torch.zeros(B * heads * Sp * 384, dtype=torch.uint8, device="cuda") for _ in range(3))
    ctx = torch.zeros(lib.cubert_split_bytes(B * S, H), dtype=torch.uint8, device="cuda")
    check(lib.cubert_op_gemm_qkv(xs.data_ptr(), ws.data_ptr(), bd.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), B, S, heads,
                                 SPLIT, tile, 0, None))
    check(lib.cubert_op_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), md.data_ptr(), ctx.data_ptr(), B, heads, S, 0.125, SPLIT,
                                  0, None))
    torch.cuda.synchronize()
    # a score is off by the projections' errors and its own 24 accumulations, relative to sum |q k|; its probability by
    # twice that; the context averages values with those probabilities, after the values' own error and S roundings
    proj = (6 * H / 16 + 2) * U * scale_in
    qk = float(torch.matmul(qkv[0].abs(), qkv[1].abs().transpose(-1, -2).contiguous()).max()) * 0.125
    dscore = 26 * U * qk + 2 * proj * float(qkv[:2].abs().sum(-1).max()) * 0.125 + 4 * U * float(sc[sc > -5000].abs().max())
    bound = float(qkv[2].abs().max()) * (2 * dscore + (S + 26) * U) + proj
    assert float((unsplit(ctx, B * S, H).cpu() - want).abs().max()) < bound


@pytest.mark.parametrize("B,S,heads", [(1, 1, 1), (2, 32, 1), (3, 33, 2), (2, 128, 1), (2, 129, 2), (1, 257, 1), (4, 300, 2), (1, 545, 1)])
def test_attention_kernels_agree(lib, B, S, heads):
    """The kernels whose four or eight waves share the keys and the one whose waves walk them, each against float64: masks that end early,
    leave out keys in the middle or hide every key, padding rows of the last block that hold numbers of their own."""
    H, Sp = heads * 64, (S + 31) // 32 * 32
    X, W, b = operands(B * Sp, 3 * H, H)
    X, W = X / X.abs().max() * 4, W * 2
    mask = np.zeros((B, Sp), np.float32)
    rng = np.random.default_rng(S)
    for i in range(B):
        if i == 1:
            mask[i, :] = -10000.0                        # no visible key: a uniform shift, softmax over all of them
        elif i == 2:
            mask[i, rng.random(Sp) < 0.5] = -10000.0
        elif i == 3:
            mask[i, 1:] = -10000.0
    mask[:, S:] = -np.inf
    xs, ws, bd, md = split(lib, X.cuda()), split(lib, W.cuda()), b.cuda(), torch.from_numpy(mask).cuda()
    q, k, v = (torch.zeros(B * heads * Sp * 384, dtype=torch.uint8, device="cuda") for _ in range(3))
    # every position of the padded blocks is written, as a longer batch before this one would have left it
    check(lib.cubert_op_gemm_qkv(xs.data_ptr(), ws.data_ptr(), bd.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), B, Sp, heads,
                                 SPLIT, 128, 0, None))
    qkv = (X.double() @ W.double().t() + b.double()).view(B, Sp, 3, heads, 64)[:, :S].permute(2, 0, 3, 1, 4)
    sc = torch.matmul(qkv[0], qkv[1].transpose(-1, -2).contiguous()) * 0.125
    want = torch.matmul(torch.softmax(sc + torch.from_numpy(mask[:, None, None, :S]).double(), -1), qkv[2]).permute(0, 2, 1, 3).reshape(B * S, H)
    scale_in = float((X.double().abs() @ W.double().abs().t() + b.double().abs()).max())
    proj = (6 * H / 16 + 2) * U * scale_in
    qk = float(torch.matmul(qkv[0].abs(), qkv[1].abs().transpose(-1, -2).contiguous()).max()) * 0.125
    # as above; where every key is masked (second sequence), a score near 10000 has an ulp of its own
    offset = torch.tensor([10000.0 if i == 1 else 0.0 for i in range(B)], dtype=torch.float64).repeat_interleave(S)[:, None]
    dscore = 26 * U * qk + 2 * proj * float(qkv[:2].abs().sum(-1).max()) * 0.125 + 4 * U * (float(sc.abs().max()) + offset)
    bound = float(qkv[2].abs().max()) * (2 * dscore + (S + 26) * U) + proj
    for variant in (1, 2, 3):
        ctx = torch.full((lib.cubert_split_bytes(B * S, H),), 0x7f, dtype=torch.uint8, device="cuda")
        check(lib.cubert_op_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), md.data_ptr(), ctx.data_ptr(), B, heads, S, 0.125, SPLIT,
                                      variant << 20, None))
        torch.cuda.synchronize()
        got = unsplit(ctx, B * S, H).cpu()
        assert ((got - want).abs() < bound).all(), variant
