"""bf16 passes of the row counts whose LayerNorm GEMMs are one round of 256 x 256 tiles (BERT-large 14336 to 16384 rows, BERT-base
18945 to 20480) and just beyond: one stream or two, and the tile, depend on the call; the bits do not.  Two layers of each model, the
library's own choice against a model held to one stream and one held to two."""
import numpy as np
import pytest

from cudabert_amd import synth, weights as W

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

BF16 = 1
DIMS = {"base": W.BertDims(layers=2, vocab=500), "large": W.BertDims(hidden=1024, layers=2, heads=16, inter=4096, vocab=500)}
HELD = {"own": None, "one": "0", "two": "1"}


@pytest.fixture(scope="module")
def pb():
    from cudabert_amd import pybert
    return pybert


@pytest.fixture(scope="module", params=["base", "large"])
def models(request, pb, tmp_path_factory):
    d = DIMS[request.param]
    path = W.export_npy_dir(W.synth_state(d, seed=3, degenerate=False), str(tmp_path_factory.mktemp("window")))
    kept = {}
    with pytest.MonkeyPatch.context() as mp:
        for name, least in HELD.items():
            mp.delenv("CUBERT_SPLIT_MIN_TOKENS", raising=False)
            if least is not None:
                mp.setenv("CUBERT_SPLIT_MIN_TOKENS", least)
            kept[name] = pb.load_model_ex(path, d.hidden, d.layers, d.heads, d.inter, precision=BF16, max_batchsize=128,
                                          max_seq_length=256)
    yield request.param, kept
    for m in kept.values():
        pb.unload_model(m)


class Pointer:
    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f4", "version": 2}


def results(pb, m, B, S):
    pb.check(pb.lib.cubert_sync(m))
    H = pb.lib.cubert_hidden_size(m)
    return [torch.as_tensor(Pointer(p(m), s), device="cuda").cpu().numpy()
            for p, s in ((pb.lib.cubert_seq_ptr, (B, S, H)), (pb.lib.cubert_pooled_ptr, (B, H)))]


SHAPES = {"large": [(128, 112), (64, 240), (33, 240), (127, 128), (128, 128), (128, 129)],
          "base": [(128, 148), (128, 152), (81, 250), (128, 160), (128, 161), (128, 170)]}


@pytest.mark.parametrize("i", range(6))
def test_same_bits_whoever_calls(pb, models, i):
    size, kept = models
    B, S = SHAPES[size][i]
    lens = np.random.default_rng(S).integers(S // 2, S + 1, size=B).astype(np.int32)
    lens[0] = S
    ids, seg, mask = synth.make_inputs(B, S, lens, vocab=500, seed=S, prune=False)
    dev = [torch.from_numpy(a).cuda() for a in (ids, seg, mask)]
    want = None
    for name, m in kept.items():
        pooled, seq, _ = pb.encode(m, ids, seg, mask, want_seq=True)
        if want is None:
            want = seq, pooled
            assert np.isfinite(seq).all()
        assert np.array_equal(seq, want[0]) and np.array_equal(pooled, want[1]), name
        for _ in range(3):                              # queued behind each other
            pb.check(pb.lib.cubert_forward_device(m, *[t.data_ptr() for t in dev], B, S))
        got = results(pb, m, B, S)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), name
        pb.check(pb.lib.cubert_forward_device_lens(m, dev[0].data_ptr(), dev[1].data_ptr(), lens.ctypes.data, B, S))
        got = results(pb, m, B, S)
        assert np.array_equal(got[0], want[0] * mask[:, :, None]) and np.array_equal(got[1], want[1]), name


@pytest.mark.parametrize("B,S,low,high", [(128, 157, 90, 140), (128, 160, 60, 160), (128, 168, 150, 159), (128, 128, 100, 128),
                                          (128, 126, 112, 120), (128, 140, 110, 120)])
def test_padding_skipped_unasked_leaves_no_trace(pb, models, B, S, low, high):
    """A pooled-only call computes the valid tokens alone.  Padded and valid rows lie inside and outside the window in turn."""
    size, kept = models
    lens = np.random.default_rng(B + S).integers(low, high + 1, size=B)
    ids, seg, mask = synth.make_inputs(B, S, lens, vocab=500, seed=S, prune=False)
    full = pb.encode(kept["one"], ids, seg, mask, want_seq=True)[0]
    for name, m in kept.items():
        assert np.array_equal(pb.encode(m, ids, seg, mask)[0], full), name
