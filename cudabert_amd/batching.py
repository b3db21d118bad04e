"""Length-bucketed batching frontend for one device.

Host-side counterpart of the reference's ``queue_manager`` / ``batch_container``
(engine.py:12-130), ``optimize_batch`` / ``Batch_Packed`` / ``Tagged_line``
(utils.py:3-60) and the ordered writer of ``Engine._engine_postprocess``
(engine.py:303-372), reduced to a single process and a single device: the
reference's reader, model and writer processes and their multiprocessing queues
become three steps of one loop.

What is kept, because it determines the (batch, seq) shapes the engine sees:

* the useful length of a line is the position of its last mask 1 plus one
  (utils.py:46-52);
* bucket edges ``[0, start, start+step, ..., end, max_seq_length]``
  (engine.py:225-232); a line goes to the first bucket whose upper edge is not
  below its length (engine.py:83-88);
* a bucket emits a batch when it holds ``batch_size`` lines, or when it is
  flushed (too many finished lines waiting for an earlier one);
* a batch is trimmed to its longest line (utils.py:3-13);
* among the buckets that have a batch ready the one holding the earliest input
  line goes first (engine.py:117-124);
* results leave in input order (engine.py:325-361).

Differences: ready batches of a bucket leave first-in first-out (the reference
pops the newest one while ranking buckets by their oldest, engine.py:58-61); a
line whose mask has no 1 at all has length 1 rather than 512; at the end of the
input the lines left in neighbouring buckets share a batch where that costs less
than a batch for each (``QueueManager.merge_rest``).
"""
from __future__ import annotations

import sys
from bisect import bisect_left, bisect_right
from collections import deque
from heapq import heappop, heappush
from itertools import accumulate
from typing import Callable, Iterable, List, Optional, Sequence

import numpy as np


# What a batch costs whatever it holds, in tokens of padding that a pass computes in the same time.  Pooled-only calls on MI355X,
# lines merged by cost with 360 / 1024 / 1536 tokens, one batch per bucket and batches filled whatever the padding beside them:
#   2000 lines of 8 to 200 tokens  BERT-large bf16  204.8 / 193.8 / 193.4 ms, 291.8 and 190.9   fp32  745 / 736 / 733 ms, 862 and 726
#   300 lines of 8 to 200          BERT-large bf16   40.3 /  35.7 /  33.3 ms, 104.4 and 28.8    fp32  126 / 115 / 113 ms, 229 and 99
#   100 lines of 8 to 64           BERT-large bf16   7.37 /  7.32 /  6.24 ms, 13.4 and 6.28     fp32  19.9 / 20.0 / 22.1 ms, 29.6 and 22.1
# From 1536 on the model whose tokens cost most (BERT-large fp32) loses; filled whatever the padding, 15 lines of 20 tokens and one
# of 512 take 7.6 ms in bf16 and 24.6 in fp32 where a batch for each length takes 2.8 and 6.3.
PASS_TOKENS = 1024


def generate_splits(max_seq_length: int, start_split: int = 50, end_split: int = 180, split_size: int = 2) -> List[int]:
    """Bucket edges, engine.py:225-232 (defaults from the reference's config comment, engine.py:196-198)."""
    edges = [0]
    edges.extend(range(start_split, end_split + split_size, split_size))
    edges.append(max_seq_length)
    return edges


class TaggedLine:
    """One tokenised input line (utils.py:33-60)."""

    __slots__ = ("num_line", "line_data", "input_ids", "input_mask", "segment_ids", "length", "output")

    def __init__(self, num_line: int, line_data, input_ids, input_mask, segment_ids):
        self.num_line = num_line
        self.line_data = line_data
        self.input_ids = np.asarray(input_ids, dtype=np.int32)
        self.input_mask = np.asarray(input_mask, dtype=np.int32)
        self.segment_ids = np.asarray(segment_ids, dtype=np.int32)
        if not (self.input_ids.shape == self.input_mask.shape == self.segment_ids.shape) or self.input_ids.ndim != 1:
            raise ValueError("input_ids, input_mask and segment_ids must be 1-D and of equal length")
        ones = (self.input_mask == 1).nonzero()[0]
        self.length = int(ones[-1]) + 1 if ones.size else 1
        self.output = None

    def get_tensor(self, index: int):
        return (self.input_ids, self.segment_ids, self.input_mask)[index]


def optimize_batch(lines: Sequence[TaggedLine]):
    """[ids, segments, mask], each int32 [len(lines), longest line] (utils.py:3-13)."""
    max_length = max(l.length for l in lines)
    batch = []
    for i in range(3):
        arr = np.empty((len(lines), max_length), dtype=np.int32)
        for j, l in enumerate(lines):
            arr[j] = l.get_tensor(i)[:max_length]
        batch.append(arr)
    return batch


class BatchPacked:
    """A batch and the lines it came from (utils.py:15-31)."""

    def __init__(self, lines_list: List[TaggedLine], tensor):
        self.lines_list = lines_list
        self.tensor = tensor
        self.output = None

    def set_output(self, output):
        self.output = output

    def write_line(self):
        for line, out in zip(self.lines_list, self.output):
            line.output = out


class BatchContainer:
    """Lines of one length bucket (engine.py:12-61)."""

    def __init__(self, base_length: int, top_length: int, batchsize: int, queue: Optional[List[tuple]] = None, index: int = 0):
        self.base_length = base_length
        self.top_length = top_length
        self.batchsize = batchsize
        self.queue = queue               # heap that every batch joins when it becomes ready: (first line, index); None: nobody asks
        self.index = index
        self.temp: List[TaggedLine] = []
        self.prepare: deque = deque()

    def put(self, line: TaggedLine):
        self.temp.append(line)
        if len(self.temp) == self.batchsize:
            self._batch()

    def _batch(self):
        if self.temp:
            self.emit(self.temp)
            self.temp = []

    def emit(self, lines: List[TaggedLine]):
        """Lines in input order; ready batches stay in the order of their first lines."""
        at = len(self.prepare)
        while at and self.prepare[at - 1].lines_list[0].num_line > lines[0].num_line:
            at -= 1
        self.prepare.insert(at, BatchPacked(lines, optimize_batch(lines)))
        if self.queue is not None:
            heappush(self.queue, (lines[0].num_line, self.index))

    def force_enqueue(self):
        self._batch()

    @property
    def min_index(self) -> int:
        return self.prepare[0].lines_list[0].num_line if self.prepare else sys.maxsize

    def pop(self) -> BatchPacked:
        return self.prepare.popleft()


class QueueManager:
    """Routes lines to their bucket and hands out ready batches (engine.py:63-130)."""

    def __init__(self, seq_length_split: Sequence[int], batchsize: int):
        if len(seq_length_split) < 2 or any(b <= a for a, b in zip(seq_length_split, seq_length_split[1:])):
            raise ValueError("bucket edges must be strictly increasing")
        self.boardlines = list(seq_length_split)
        self.batchsize = batchsize
        # (first line, bucket) of every ready batch.  The loop asks for one after every line it reads, and the device has nothing
        # to do meanwhile: 61 ms of host time for a file of 2000 lines when every bucket was looked at each time and a line's
        # bucket searched edge by edge, 29 with the heap and the bisection.
        self.queue: List[tuple] = []
        self.containers = [BatchContainer(a, b, batchsize, self.queue, q)
                           for q, (a, b) in enumerate(zip(self.boardlines, self.boardlines[1:]))]

    def put(self, line: TaggedLine):
        if line.length > self.boardlines[-1]:
            raise ValueError("line %d has length %d, above max_seq_length %d" %
                             (line.num_line, line.length, self.boardlines[-1]))
        self.containers[bisect_left(self.boardlines, line.length, 1) - 1].put(line)

    def force_enqueue(self):
        for c in self.containers:
            c.force_enqueue()

    def merge_rest(self):
        """End of the input: the lines still waiting, in order of length, in the batches that cost least, where a batch costs its
        tokens, padding included, and ``PASS_TOKENS``, and ends at a bucket edge or full.  (A bucket is a few tokens wide and is
        left with a few dozen lines, a batch on which the device is as good as idle.  Padding counts in full: the engine skips
        it in some calls only, and the callback may be any.)  Never more batches than one per bucket, and never more tokens
        than ``PASS_TOKENS`` for each batch less."""
        rests = [c for c in self.containers if c.temp]
        lines = sorted((l for c in rests for l in c.temp), key=lambda l: l.length)      # bucket after bucket
        edges = list(accumulate(len(c.temp) for c in rests))
        best = [(0, 0)] + [None] * len(lines)         # the first n lines: least cost, and where their last batch begins
        for begin in range(len(lines)):
            if best[begin] is None:
                continue
            full = begin + self.batchsize
            ends = [e for e in edges[bisect_right(edges, begin):] if e < full]
            for end in ends + [min(full, len(lines))]:
                cost = best[begin][0] + (end - begin) * lines[end - 1].length + PASS_TOKENS
                if best[end] is None or cost < best[end][0]:
                    best[end] = (cost, begin)
        end = len(lines)
        while end:
            begin = best[end][1]
            rests[bisect_left(edges, end)].emit(sorted(lines[begin:end], key=lambda l: l.num_line))
            end = begin
        for c in rests:
            c.temp = []

    def ready(self) -> int:
        return sum(len(c.prepare) for c in self.containers)

    def get(self) -> Optional[BatchPacked]:
        """The ready batch that holds the earliest input line, or None."""
        while self.queue:
            num_line, q = heappop(self.queue)
            # (a batch may have been taken from its bucket directly)
            if self.containers[q].min_index == num_line:
                return self.containers[q].pop()
        return None


class OrderedWriter:
    """Releases per-line results in input order (engine.py:303-372)."""

    def __init__(self, sink: Callable[[object], None]):
        self.sink = sink
        self.next_line = 0
        self.waiting = {}

    def add(self, batch: BatchPacked):
        batch.write_line()
        for line in batch.lines_list:
            if line.num_line < self.next_line or line.num_line in self.waiting:
                raise RuntimeError("line index %d is written twice" % line.num_line)
            self.waiting[line.num_line] = line
        while self.next_line in self.waiting:
            self.sink(self.waiting.pop(self.next_line))
            self.next_line += 1

    @property
    def backlog(self) -> int:
        return len(self.waiting)


class Engine:
    """Single-device ``Engine.run`` (engine.py:377-403): tokenise -> bucket -> encode -> ordered output.

    tokenize(max_seq_length, line, index) -> (index, line_data, input_ids, input_mask, segment_ids)
        as the reference's ``tokenlizer_line`` callback (engine.py:291-292).
    encode([ids, segments, mask]) -> per-line outputs [batch, ...]   (``Cuda_BERT.encode`` plus,
        if wanted, the fine-tune layer; engine.py:258-260).
    output(line_data, line_output) -> what ``sink`` receives for the line (engine.py:338-339).
    """

    def __init__(self, encode, tokenize, output=lambda data, out: out, max_seq_length: int = 200,
                 batch_size: int = 128, start_split: int = 50, end_split: int = 180, split_size: int = 2,
                 alert_size: int = 1000000):
        self.encode, self.tokenize, self.output = encode, tokenize, output
        self.max_seq_length, self.batch_size, self.alert_size = max_seq_length, batch_size, alert_size
        self.splits = generate_splits(max_seq_length, start_split, end_split, split_size)
        self.batch_shapes: List[tuple] = []          # (batch, seq) of every batch sent to the device

    def _drain(self, manager: QueueManager, writer: OrderedWriter):
        while True:
            batch = manager.get()
            if batch is None:
                return
            self.batch_shapes.append(batch.tensor[0].shape)
            batch.set_output(self.encode(batch.tensor))
            writer.add(batch)

    def run(self, lines: Iterable[str], sink: Callable[[object], None]):
        manager = QueueManager(self.splits, self.batch_size)
        writer = OrderedWriter(lambda line: sink(self.output(line.line_data, line.output)))
        for index, text in enumerate(lines):
            manager.put(TaggedLine(*self.tokenize(self.max_seq_length, text, index)))
            self._drain(manager, writer)
            if writer.backlog > self.alert_size:      # finished lines pile up behind a half-full bucket
                manager.force_enqueue()
                self._drain(manager, writer)
        manager.merge_rest()
        self._drain(manager, writer)
        if writer.backlog:
            raise RuntimeError("%d results were never released" % writer.backlog)
