"""Performance cases of the encoder: what a user of the library has it do, over the sizes it is used at.

The ranges: BERT-base and BERT-large, both precisions (float32 is the library's default), batches of one line up to 128,
lines of a few tokens up to the position table's 512, and the ways in:

* ``bert``         pooled output on the host, the serving engine's call (``Cuda_BERT.encode``)
* ``encode``       pooled output, sequence output and class probabilities on the host
* ``inference``    host inputs, sequence and pooled output left in device memory
* ``device``       inputs, sequence output, pooled output and class probabilities in device memory
* ``device_lens``  the same on the valid tokens only
* ``lines``        tokenised lines of a text file through the length-bucketed frontend, results in input order

Token ids, segments and masks look like the frontend's: valid lengths uniform in a range, one line of a batch as long as the
batch is wide, segment 1 on the second half of a line, padding masked.  Weights are a seeded synthetic checkpoint; a model is
loaded once per process, as a serving program does, and used by every case of its size and precision.
"""
import os
import tempfile

import numpy as np
import torch

from cudabert_amd import batching, pybert
from cudabert_amd import weights as W

DIMS = {"base": W.BASE, "large": W.LARGE}
CAPACITY = (128, 512)                   # largest batch and line length a model is loaded for
PRECISIONS = {"fp32": pybert.F32, "bf16": pybert.BF16}
WEIGHT_SEED = 20240
FIRST_ID = 1000                         # word pieces; lower ids are special tokens

_models = {}


def _model(size, precision):
    key = (size, precision)
    if key not in _models:
        dims = DIMS[size]
        with tempfile.TemporaryDirectory() as d:
            W.export_npy_dir(W.synth_state(dims, seed=WEIGHT_SEED, degenerate=False), d)
            _models[key] = pybert.load_model_ex(d, dims.hidden, dims.layers, dims.heads, dims.inter,
                                                precision=PRECISIONS[precision], max_batchsize=CAPACITY[0],
                                                max_seq_length=CAPACITY[1])
    return _models[key]


def _case(name, size, precision, entry, batch, seq, shortest, short_share=0.0):
    c = {"size": size, "precision": precision, "entry": entry, "batch": batch, "seq": seq, "shortest": shortest,
         "short_share": short_share}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one short query, the smallest call a service makes (odd length)
        _case("query_base_bf16", "base", "bf16", "bert", 1, 17, 17),
        # one full-length line: the latency figure of the benchmark
        _case("line_large_bf16", "large", "bf16", "bert", 1, 200, 200),
        # a handful of lines, the benchmark's other latency figure
        _case("few_large_bf16", "large", "bf16", "bert", 8, 200, 200),
        # what a length bucket hands over when a file runs out: an uneven number of lines of an odd length
        _case("bucket_large_bf16", "large", "bf16", "bert", 23, 77, 70),
        # a batch of base-size lines with everything a downstream head may want, kept on the device
        _case("batch_base_bf16", "base", "bf16", "device", 128, 128, 64),
        # the headline: a full batch of the large model, sequence output included
        _case("batch_large_bf16", "large", "bf16", "device", 128, 200, 100),
        # long documents, most of them short: only valid tokens are computed
        _case("documents_large_bf16", "large", "bf16", "device_lens", 64, 512, 32, 0.7),
        # a file of lines of mixed length through the frontend
        _case("file_large_bf16", "large", "bf16", "lines", 2000, 200, 8),
        # float32, the default precision: one line, a few lines with every output on the host, long lines, a full batch
        _case("line_large_fp32", "large", "fp32", "bert", 1, 128, 128),
        _case("few_base_fp32", "base", "fp32", "encode", 8, 128, 32),
        _case("long_base_fp32", "base", "fp32", "inference", 16, 512, 300),
        _case("batch_large_fp32", "large", "fp32", "bert", 128, 200, 100),
    ]


def _cost(case):
    """Relative time of a case: float32 matrix arithmetic takes about ten times as long as bf16."""
    return work(case)["flops"] * (10.0 if case["precision"] == "fp32" else 1.0)


def draw(rng):
    limit = max(_cost(c) for c in listed())
    most = max(work(c)["flops"] for c in listed())
    while True:
        size = rng.choice(["base", "large"])
        precision = rng.choice(["fp32", "bf16"])
        entry = rng.choice(["bert", "bert", "encode", "inference", "device", "device_lens", "lines"])
        seq = int(round(8 * (512 / 8) ** rng.random()))
        if entry == "lines":
            seq = max(seq, 64)
            batch = int(round(100 * (2000 / 100) ** rng.random()))
        else:
            batch = int(round(128 ** rng.random()))
        shortest = max(1, int(round(seq * rng.uniform(0.1, 1.0))))
        case = _case(None, size, precision, entry, batch, seq, shortest, round(rng.choice([0.0, 0.0, rng.random()]), 2))
        # every output on the host: the copy of the sequence output stays a part of the call, not the whole of it
        if entry == "encode" and batch * seq > 4096:
            continue
        if _cost(case) <= limit and work(case)["flops"] <= most:
            return case


def _lengths(case, rng):
    """Valid length of every line: uniform in shortest .. seq, a share of the lines in the lowest quarter of that range;
    one line is seq long."""
    lo, hi, n = case["shortest"], case["seq"], case["batch"]
    lens = rng.integers(lo, hi + 1, size=n)
    short = rng.random(n) < case["short_share"]
    lens = np.where(short, rng.integers(lo, lo + (hi - lo) // 4 + 1, size=n), lens)
    lens[int(rng.integers(0, n))] = hi
    return lens.astype(np.int32)


def _inputs(case, rng, lens):
    n, seq, vocab = case["batch"], case["seq"], DIMS[case["size"]].vocab
    col = np.arange(seq)[None, :]
    valid = col < lens[:, None]
    ids = np.where(valid, rng.integers(FIRST_ID, vocab, size=(n, seq)), 0).astype(np.int32)
    seg = (valid & (col >= lens[:, None] // 2)).astype(np.int32)
    return ids, seg, valid.astype(np.int32)


class _DevicePointer:
    """A float32 result of the library in device memory, for torch.as_tensor."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f4", "version": 2}


def _view(ptr, *shape):
    return torch.as_tensor(_DevicePointer(ptr, shape), device="cuda")


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    model = _model(case["size"], case["precision"])
    lens = _lengths(case, rng)
    ids, seg, mask = _inputs(case, rng, lens)
    state = {"entry": case["entry"], "model": model, "B": case["batch"], "S": case["seq"],
             "H": DIMS[case["size"]].hidden, "C": int(pybert.lib.cubert_num_classes(model))}
    if case["entry"] in ("device", "device_lens"):
        state.update(ids=torch.from_numpy(ids).cuda(), seg=torch.from_numpy(seg).cuda(), mask=torch.from_numpy(mask).cuda(),
                     lens=lens)
    else:
        state.update(ids=ids, seg=seg, mask=mask)
    if case["entry"] == "bert":
        state["out"] = np.empty((case["batch"], state["H"]), np.float32)
    if case["entry"] == "lines":
        def encode(tensor):
            out = np.empty((tensor[0].shape[0], state["H"]), np.float32)
            pybert.bert(model, out, tensor[0], tensor[1], tensor[0].shape[0], tensor[0].shape[1], tensor[2])
            return out

        def tokenize(max_seq_length, line, index):
            return index, line, ids[line], mask[line], seg[line]

        state["engine"] = batching.Engine(encode, tokenize, max_seq_length=case["seq"], batch_size=128,
                                          end_split=min(180, case["seq"] - 2))
    return state


def run(state):
    entry, model, B, S, H = state["entry"], state["model"], state["B"], state["S"], state["H"]
    lib = pybert.lib
    if entry == "bert":
        pybert.bert(model, state["out"], state["ids"], state["seg"], B, S, state["mask"])
        return state["out"]
    if entry == "encode":
        return pybert.encode(model, state["ids"], state["seg"], state["mask"], want_seq=True, want_cls=True)
    if entry == "inference":
        r = pybert.inference(model, state["ids"], state["seg"], B, S, state["mask"])
        return _view(r.tensor, B, S, H), _view(r.Pooled_Output, B, H)
    if entry == "lines":
        rows = []
        state["engine"].run(range(B), rows.append)
        return np.stack(rows)
    if entry == "device":
        pybert.check(lib.cubert_forward_device(model, state["ids"].data_ptr(), state["seg"].data_ptr(),
                                               state["mask"].data_ptr(), B, S))
    else:
        pybert.check(lib.cubert_forward_device_lens(model, state["ids"].data_ptr(), state["seg"].data_ptr(),
                                                    state["lens"].ctypes.data, B, S))
    pybert.check(lib.cubert_classify(model))
    return (_view(lib.cubert_seq_ptr(model), B, S, H), _view(lib.cubert_pooled_ptr(model), B, H),
            _view(lib.cubert_cls_ptr(model), B, state["C"]))


def work(case):
    """Floating-point operations of the encoder's matrix products and attention, and the bytes of weights, inputs and results.

    Tokens: the valid ones, or all of them where the call returns a sequence output on the padding too.  A call that returns
    pooled outputs only needs, in the last layer, keys and values of every token and the rest of the first tokens alone."""
    d = DIMS[case["size"]]
    H, L, I, n, seq = d.hidden, d.layers, d.inter, case["batch"], case["seq"]
    lo = case["shortest"]
    mean = (lo + seq) / 2
    short = (lo + lo + (seq - lo) // 4) / 2
    mean = case["short_share"] * short + (1 - case["short_share"]) * mean
    padded = case["entry"] in ("encode", "inference", "device")
    pooled_only = case["entry"] in ("bert", "lines")
    tokens = n * (seq if padded else mean)
    keys = mean                                              # keys a query attends to
    layer = tokens * (2 * H * (4 * H + 2 * I) + 4 * keys * H)
    flops = L * layer
    if pooled_only:
        flops -= layer - tokens * 2 * H * 2 * H - n * (2 * H * (2 * H + 2 * I) + 4 * keys * H)
    flops += n * 2 * H * H
    es = 2 if case["precision"] == "bf16" else 4
    weights = (L * (4 * H * H + 2 * H * I) + H * H) * es + L * (9 * H + I) * 4
    embeddings = min(n * mean, d.vocab) * H * 4
    results = n * H * 4 + (0 if pooled_only else n * seq * H * 4)
    return {"bytes": weights + embeddings + 3 * 4 * n * seq + results, "flops": flops}


def tolerance(case):
    """About four times what correct implementations differ by.  float32: the path against a float64 restatement of the model,
    1.4e-6 in 2-norm and 7.6e-6 at the worst element (two dozen layers).  bf16: the path against itself with its float32
    sums in another order (K of the short products not split, keys of the attention split), 4.5e-3 and 4.4e-2: a sum that
    lands on the other side of a bf16 rounding sends the rest of the pass down another rounding path."""
    if case["precision"] == "fp32":
        return {"rel": 6e-6, "max": 3e-5}
    return {"rel": 1.8e-2, "max": 0.18}
