"""bf16 GEMMs on operands in the units layout (MFMA operand order), at the edges of tiles, row blocks and K steps.

Bounds: operands are bf16 on both sides, so a float32 result differs from float64 by its K / 16 float32 accumulations and a
few additions, (K / 16 + 6) 2^-24 sum |x w| at the worst; a bf16 result by half a bf16 step more, and GELU by the 7e-5 of its
polynomial."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
U = 2.0 ** -24
PACKED = {"X": 1, "W": 2, "Y": 4}
UNITS = {"X": 128, "W": 1 << 24, "Y": 1 << 25}
SKINNY = (97, 98)


@pytest.fixture(scope="module")
def lib():
    from cudabert_amd import pybert
    lib = pybert.lib
    lib.cubert_units_offset.argtypes = [ctypes.c_int] * 3
    lib.cubert_units_offset.restype = ctypes.c_size_t
    return lib


def check(rc):
    from cudabert_amd import pybert
    pybert.check(rc)


def index(R, K, units):
    """bf16 index of element (r, k) in the packed layout or its units form."""
    r, k = np.arange(R)[:, None], np.arange(K)[None, :]
    block = ((r >> 8) * (K // 32) + (k >> 5)) * 8192
    if units:
        return block + ((r >> 5) & 7) * 1024 + ((k >> 4) & 1) * 512 + ((k >> 3) & 1) * 256 + (r & 31) * 8 + (k & 7)
    return block + (r & 255) * 32 + ((((k >> 3) & 3) ^ ((r >> 2) & 3)) << 3) + (k & 7)


def pack(lib, a, units):
    R, K = a.shape
    buf = torch.zeros(lib.cubert_packed_bytes(R, K * 2) // 2, dtype=torch.bfloat16)
    buf[torch.from_numpy(index(R, K, units))] = a
    return buf.cuda()


def test_units_offset_formula(lib):
    idx = index(300, 128, True)
    for r, k in ((0, 0), (1, 9), (17, 40), (255, 127), (256, 0), (299, 77)):
        assert lib.cubert_units_offset(r, k * 2, 256) == idx[r, k] * 2
    assert len(np.unique(idx)) == idx.size


def operands(M, N, K):
    g = torch.Generator().manual_seed(7)
    X = torch.randn(M, K, generator=g).to(torch.bfloat16)
    W = (torch.randn(N, K, generator=g) * 0.05).to(torch.bfloat16)
    b = torch.randn(N, generator=g)
    want = X.double() @ W.double().t() + b.double()
    scale = X.double().abs() @ W.double().abs().t() + b.double().abs()
    return X, W, b, want, scale


@pytest.mark.parametrize("xu,wu", [(True, True), (False, True), (True, False)])
@pytest.mark.parametrize("tile,M,N,K", [(64, 1, 32, 64), (64, 70, 96, 192), (192, 129, 160, 64), (128, 200, 320, 128), (256, 257, 288, 256),
                                        (384, 130, 288, 192), (385, 130, 288, 256), (97, 1, 32, 128), (97, 130, 96, 192), (98, 65, 200, 256)])
def test_float32_result(lib, tile, M, N, K, xu, wu):
    if tile in SKINNY and not (xu and wu):
        pytest.skip("both operands in units")
    X, W, b, want, scale = operands(M, N, K)
    R = torch.randn(M, N, generator=torch.Generator().manual_seed(2))
    xp, wp, bd, Rd = pack(lib, X, xu), pack(lib, W, wu), b.cuda(), R.cuda()
    Y = torch.full((2, M, N), float("nan"), device="cuda")
    flags = 3 | (UNITS["X"] if xu else 0) | (UNITS["W"] if wu else 0)
    check(lib.cubert_op_gemm_residual(xp.data_ptr(), wp.data_ptr(), bd.data_ptr(), Rd.data_ptr(), Y.data_ptr(), M, N, K, K, 1, tile, flags, None))
    torch.cuda.synchronize()
    assert ((Y[0].double().cpu() - want - R.double()).abs() <= (K / 16 + 6) * U * (scale + R.double().abs())).all()
    assert torch.isnan(Y[1]).all()


@pytest.mark.parametrize("tile,M,N,K", [(64, 1, 32, 64), (64, 70, 96, 192), (192, 129, 160, 64), (128, 200, 320, 128), (256, 300, 288, 256),
                                        (384, 130, 288, 192), (385, 130, 288, 256), (97, 1, 32, 128), (97, 130, 96, 192), (98, 65, 256, 256)])
def test_gelu_result_in_units(lib, tile, M, N, K):
    X, W, b, want, scale = operands(M, N, K)
    xp, wp, bd = pack(lib, X, True), pack(lib, W, True), b.cuda()
    Y = torch.zeros(lib.cubert_packed_bytes(M, N * 2) // 2, dtype=torch.bfloat16, device="cuda")
    check(lib.cubert_op_gemm(xp.data_ptr(), wp.data_ptr(), bd.data_ptr(), Y.data_ptr(), M, N, K, K, 1, 1, 1, tile, 7 | sum(UNITS.values()), None))
    torch.cuda.synchronize()
    got = Y.cpu()[torch.from_numpy(index(M, N, True))].double()
    want = 0.5 * want * (1 + torch.erf(want / np.sqrt(2.0)))
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 7e-5 + 1.13 * (K / 16 + 6) * U * scale).all()


@pytest.mark.parametrize("B,S,heads", [(1, 5, 2), (2, 33, 2), (3, 200, 3)])
@pytest.mark.parametrize("tile", SKINNY)
def test_skinny_qkv_matches_the_staged_tile(lib, tile, B, S, heads):
    """Q, K, V rows of the tile without a staged loop against the 64 tile's: same products, sums over K in another order."""
    H = heads * 64
    X, W, b, want, scale = operands(B * S, 3 * H, H)
    xp, wp, bd = pack(lib, X, True), pack(lib, W, True), b.cuda()
    out = [torch.zeros(B, heads, S, 64, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
    check(lib.cubert_op_gemm_qkv(xp.data_ptr(), wp.data_ptr(), bd.data_ptr(), *[t.data_ptr() for t in out], B, S, heads, 1, tile,
                                 3 | UNITS["X"] | UNITS["W"] | 32, None))
    torch.cuda.synchronize()
    for i, t in enumerate(out):
        ref = want[:, i * H:(i + 1) * H].view(B, S, heads, 64).permute(0, 2, 1, 3)
        lim = scale[:, i * H:(i + 1) * H].view(B, S, heads, 64).permute(0, 2, 1, 3)
        assert ((t.double().cpu() - ref).abs() <= 2.0 ** -8 * ref.abs() + (H / 16 + 6) * U * lim).all()


@pytest.fixture(scope="module")
def two_layers(tmp_path_factory):
    import dataclasses
    from cudabert_amd import pybert
    from cudabert_amd import weights as W
    dims = dataclasses.replace(W.BASE, layers=2, vocab=500)
    d = str(tmp_path_factory.mktemp("two_layers"))
    W.export_npy_dir(W.bf16_representable(W.synth_state(dims, seed=3, degenerate=False)), d)
    m = pybert.load_model_ex(d, dims.hidden, dims.layers, dims.heads, dims.inter, precision=1, max_batchsize=2, max_seq_length=300)
    yield m, W.load_npy_dir(d), dims
    pybert.unload_model(m)


@pytest.mark.parametrize("B,S", [(1, 1), (1, 17), (1, 64), (1, 65), (1, 128), (1, 129), (1, 256), (1, 257), (2, 129)])
def test_rows_at_which_the_model_changes_layout_and_tile(two_layers, B, S):
    """Row counts at the edges of 32- and 256-row blocks and at the line where the plan changes its costs (257); eager and replayed pass against the float32
    oracle at the bf16 mode's tolerance, 3e-2."""
    from cudabert_amd import pybert, synth
    from oracle import bert_oracle as O
    m, npy, dims = two_layers
    ids, seg, mask = synth.make_inputs(B, S, np.full(B, S), vocab=dims.vocab, seed=S, prune=False)
    seq_ref, pooled_ref = O.forward_torch(npy, dims.heads, ids, seg, mask)
    first = None
    for _ in range(4):
        pooled, seq, _ = pybert.encode(m, ids, seg, mask, want_seq=True)
        assert np.abs(seq - seq_ref).max() < 3e-2 and np.abs(pooled - pooled_ref).max() < 3e-2
        first = seq if first is None else first
        assert np.array_equal(seq, first)
