"""Bit identity at the default settings, where split K and the skinny tiles regroup sums by a row count: the routes of one
batch that compute fewer rows (the first tokens alone in the last layer, the valid tokens alone) decide on the same rows.
Two layers of BERT-base, BERT-large and a small model; the row counts lie on both sides of the changes of plan (float32,
BERT-base, 1300 rows and small, 2560: skinny tiles that do not split K)."""
import numpy as np
import pytest

from cudabert_amd import synth, weights as W

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")

F32, BF16 = 0, 1
DIMS = {"small": W.BertDims(hidden=128, layers=2, heads=2, inter=512, vocab=500), "base": W.BertDims(layers=2, vocab=500), "large": W.BertDims(hidden=1024, layers=2, heads=16, inter=4096, vocab=500)}


@pytest.fixture(scope="module")
def pb():
    from cudabert_amd import pybert
    return pybert


@pytest.fixture(scope="module")
def dirs(tmp_path_factory):
    root = tmp_path_factory.mktemp("two_layers")
    return {size: W.export_npy_dir(W.synth_state(d, seed=3, degenerate=False), str(root / size)) for size, d in DIMS.items()}


@pytest.fixture(scope="module")
def models(pb, dirs):
    kept = {}

    def get(size, precision):
        if (size, precision) not in kept:
            d = DIMS[size]
            kept[size, precision] = pb.load_model_ex(dirs[size], d.hidden, d.layers, d.heads, d.inter, precision=precision,
                                                     max_batchsize=64, max_seq_length=512, graph_max_tokens=8192)
        return kept[size, precision]
    yield get
    for m in kept.values():
        pb.unload_model(m)


SIZES = [("small", F32), ("small", BF16), ("base", F32), ("large", F32), ("base", BF16), ("large", BF16)]


@pytest.mark.parametrize("B,S", [(1, 17), (4, 32), (3, 67), (8, 128), (10, 130), (16, 128), (20, 128), (20, 150), (31, 200), (40, 200), (64, 200)])
@pytest.mark.parametrize("size,precision", SIZES)
def test_pooled_only_call_has_the_bits_of_the_full_pass(pb, models, size, precision, B, S):
    m = models(size, precision)
    ids, seg, _ = synth.make_inputs(B, S, [S] * B, vocab=500, seed=B)
    full, _, cls_full = pb.encode(m, ids, seg, None, want_seq=True, want_cls=True)
    pooled, _, cls = pb.encode(m, ids, seg, None, want_cls=True)
    assert np.array_equal(pooled, full) and np.array_equal(cls, cls_full)


@pytest.mark.parametrize("B,S,low,high", [(42, 200, 20, 60), (60, 150, 20, 150), (64, 150, 60, 150), (64, 200, 20, 70), (64, 512, 32, 120),
                                          (64, 512, 8, 20)])
@pytest.mark.parametrize("size,precision", SIZES)
def test_padding_skipped_unasked_leaves_no_trace(pb, models, size, precision, B, S, low, high):
    """More than 8192 tokens with padding: a pooled-only call computes the valid tokens alone, one that returns the sequence
    output the padded batch."""
    m = models(size, precision)
    lens = np.random.default_rng(B + S).integers(low, high + 1, size=B)
    ids, seg, mask = synth.make_inputs(B, S, lens, vocab=500, seed=S, prune=False)
    full, _, cls_full = pb.encode(m, ids, seg, mask, want_seq=True, want_cls=True)
    pooled, _, cls = pb.encode(m, ids, seg, mask, want_cls=True)
    assert np.array_equal(pooled, full) and np.array_equal(cls, cls_full)
