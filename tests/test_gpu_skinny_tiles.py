"""GEMM tiles whose eight waves share K, at the edges of what the host hands to them: tile counts that the eight XCDs do not share
evenly (or that leave some without a tile), K steps that the waves of all parts do not, numbers of parts that are no power of two,
rows past a 256-row block, features that end inside a tile.

Bounds as in the tests of the two operand layouts: K / 16 float32 accumulations (six of them per float32 product of split operands)
and a few additions against float64."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

import test_gpu_f32_split as f32  # noqa: E402
import test_gpu_units_layout as b16  # noqa: E402
from test_gpu_f32_split import lib as lib  # noqa: E402,F401

TILES = (95, 96, 97, 98)
U = 2.0 ** -24
SHAPES = [(1, 32, 64, 1), (17, 264, 512, 3), (33, 72, 1088, 5), (65, 328, 192, 1), (300, 96, 1088, 1), (257, 1160, 256, 2)]


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K,splits", SHAPES)
@pytest.mark.parametrize("split_operands", [False, True])
def test_float32_result_in_parts(lib, tile, M, N, K, splits, split_operands):  # noqa: F811
    steps = K // (16 if split_operands else 32)
    if 4 * splits > steps:
        pytest.skip("at least four K steps a part")
    X, W, b = (f32.operands(M, N, K) if split_operands else b16.operands(M, N, K))[:3]
    R = torch.randn(M, N, generator=torch.Generator().manual_seed(2))
    want = X.double() @ W.double().t() + b.double() + R.double()
    scale = X.double().abs() @ W.double().abs().t() + b.double().abs() + R.double().abs()
    if split_operands:
        xp, wp, elt, flags = f32.split(lib, X.cuda()), f32.split(lib, W.cuda()), f32.SPLIT, 0
    else:
        xp, wp, elt, flags = b16.pack(lib, X, True), b16.pack(lib, W, True), 1, 3 | b16.UNITS["X"] | b16.UNITS["W"]
    bd, Rd = b.cuda(), R.cuda()
    Y = torch.full((splits + 1, M, N), float("nan"), device="cuda")
    f32.check(lib.cubert_op_gemm_residual(xp.data_ptr(), wp.data_ptr(), bd.data_ptr(), Rd.data_ptr(), Y.data_ptr(), M, N, K, K, elt, tile,
                                          flags | (splits << 8 if splits > 1 else 0), None))
    torch.cuda.synchronize()
    assert torch.isnan(Y[splits]).all()                  # nothing past the last part
    products = 6 if split_operands else 1
    assert ((Y[:splits].double().sum(0).cpu() - want).abs() <= (products * K / 16 + 6 + splits) * U * scale).all()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("B,S,heads", [(1, 1, 1), (3, 11, 1), (2, 150, 3)])
def test_qkv_rows(lib, tile, B, S, heads):  # noqa: F811
    """Token and head of every row from multiplications instead of divisions (a line of one token: no division at all)."""
    H = max(heads, 2) * 64
    X, W, b, want, scale = b16.operands(B * S, 3 * H, H)
    xp, wp, bd = b16.pack(lib, X, True), b16.pack(lib, W, True), b.cuda()
    heads = H // 64
    out = [torch.zeros(B, heads, S, 64, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
    f32.check(lib.cubert_op_gemm_qkv(xp.data_ptr(), wp.data_ptr(), bd.data_ptr(), *[t.data_ptr() for t in out], B, S, heads, 1, tile,
                                     3 | b16.UNITS["X"] | b16.UNITS["W"] | 32, None))
    torch.cuda.synchronize()
    for i, t in enumerate(out):
        ref = want[:, i * H:(i + 1) * H].view(B, S, heads, 64).permute(0, 2, 1, 3)
        lim = scale[:, i * H:(i + 1) * H].view(B, S, heads, 64).permute(0, 2, 1, 3)
        assert ((t.double().cpu() - ref).abs() <= 2.0 ** -8 * ref.abs() + (H / 16 + 6) * U * lim).all()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N", [(129, 256), (256, 320)])
@pytest.mark.parametrize("split_operands", [False, True])
def test_xcd_partitions_give_the_same_bits(lib, tile, M, N, split_operands):  # noqa: F811
    """Who computes a tile is all that a partition changes; one that does not divide the grid is left out."""
    K = 256
    X, W, b = (f32.operands(M, N, K) if split_operands else b16.operands(M, N, K))[:3]
    if split_operands:
        xp, wp, elt, flags = f32.split(lib, X.cuda()), f32.split(lib, W.cuda()), f32.SPLIT, 0
    else:
        xp, wp, elt, flags = b16.pack(lib, X, True), b16.pack(lib, W, True), 1, 3 | b16.UNITS["X"] | b16.UNITS["W"]
    bd, out = b.cuda(), []
    for partition in (-1, 0, 2, 4):
        Y = torch.full((2, M, N), float("nan"), device="cuda")
        f32.check(lib.cubert_op_gemm(xp.data_ptr(), wp.data_ptr(), bd.data_ptr(), Y.data_ptr(), M, N, K, K, elt, 0, 0, tile,
                                     flags | ((partition + 1) << 16) | 2 << 8, None))
        torch.cuda.synchronize()
        assert not torch.isnan(Y).any()
        out.append(Y)
    assert all(torch.equal(out[0], y) for y in out[1:])


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 9, 13])
@pytest.mark.parametrize("split_operands", [False, True])
def test_steps_of_a_wave(lib, tile, steps, split_operands):  # noqa: F811
    """Every number of K steps that a wave keeps in flight, and more than those; some waves have a step less."""
    K = 128 * steps - 48 if split_operands else 256 * steps - 64
    M, N = 40, 72
    X, W, b = (f32.operands(M, N, K) if split_operands else b16.operands(M, N, K))[:3]
    want = X.double() @ W.double().t() + b.double()
    scale = X.double().abs() @ W.double().abs().t() + b.double().abs()
    if split_operands:
        xp, wp, elt, flags = f32.split(lib, X.cuda()), f32.split(lib, W.cuda()), f32.SPLIT, 0
    else:
        xp, wp, elt, flags = b16.pack(lib, X, True), b16.pack(lib, W, True), 1, 3 | b16.UNITS["X"] | b16.UNITS["W"]
    bd = b.cuda()
    Y = torch.full((M, N), float("nan"), device="cuda")
    f32.check(lib.cubert_op_gemm(xp.data_ptr(), wp.data_ptr(), bd.data_ptr(), Y.data_ptr(), M, N, K, K, elt, 0, 0, tile, flags, None))
    torch.cuda.synchronize()
    assert ((Y.double().cpu() - want).abs() <= ((6 if split_operands else 1) * K / 16 + 7) * U * scale).all()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K", [(1, 32, 128), (33, 96, 192), (130, 160, 512), (65, 224, 256)])
def test_gelu_in_both_layouts(lib, tile, M, N, K):  # noqa: F811
    """Features and rows that end inside a tile and inside a unit; the 32 x 32 tile leaves half of the threads without a result of their own."""
    b16.test_gelu_result_in_units(lib, tile, M, N, K)
    f32.test_gelu_result_is_the_next_split_operand(lib, tile, M, N, K)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("B,S,heads", [(1, 1, 1), (3, 45, 2), (2, 129, 3)])
def test_split_qkv_and_attention(lib, tile, B, S, heads):  # noqa: F811
    f32.test_qkv_projection_and_attention(lib, B, S, heads, tile)


def test_transposed_values(lib, tmp_path, monkeypatch):  # noqa: F811
    """Lines beyond 512 positions, whose V is stored transposed: a narrow model's QKV takes a skinny tile there (tests/test_gemm_plans.py).  Against the same
    model with sums over K in one piece, which takes the staged tile: bf16 results that differ by roundings of 2^-8, carried through one layer."""
    import dataclasses
    import numpy as np
    from cudabert_amd import pybert, synth
    from cudabert_amd import weights as Wt
    from oracle import bert_oracle as O
    dims = dataclasses.replace(Wt.BASE, hidden=256, heads=4, inter=1024, layers=1, vocab=500, max_pos=600)
    d = str(tmp_path)
    Wt.export_npy_dir(Wt.bf16_representable(Wt.synth_state(dims, seed=3, degenerate=False)), d)
    npy = Wt.load_npy_dir(d)
    out = {}
    for S in (513, 521, 544):
        ids, seg, mask = synth.make_inputs(1, S, np.full(1, S), vocab=dims.vocab, seed=S, prune=False)
        seq_ref, _ = O.forward_torch(npy, dims.heads, ids, seg, mask)
        for split in ("1", "0"):
            monkeypatch.setenv("CUBERT_SPLIT_K", split)
            m = pybert.load_model_ex(d, dims.hidden, dims.layers, dims.heads, dims.inter, precision=1, max_batchsize=1, max_seq_length=600)
            out[split] = pybert.encode(m, ids, seg, mask, want_seq=True)[1]
            pybert.unload_model(m)
            assert np.abs(out[split] - seq_ref).max() < 3e-2
        rms = np.sqrt((seq_ref ** 2).mean())
        assert np.sqrt(((out["1"] - out["0"]) ** 2).mean()) < 2.0 ** -8 * rms
