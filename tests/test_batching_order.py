"""The ready batch with the earliest line goes first, however the batches became ready and whoever took some of them."""
import copy
import random

import numpy as np
import pytest

from cudabert_amd import batching as Bt


def line(num, length, width=40):
    mask = (np.arange(width) < length).astype(np.int32)
    return Bt.TaggedLine(num, None, mask * (num + 1), mask, mask * 0)


@pytest.mark.parametrize("seed", range(6))
def test_earliest_line_first(seed):
    rng = random.Random(seed)
    qm = Bt.QueueManager([2, 8, 9, 16, 40], batchsize=3)       # (a line of 1 belongs to the first bucket as well)
    taken = 0
    for num in range(400):
        qm.put(line(num, rng.choice([1, 2, 8, 9, 10, 16, 17, 40])))
        step = rng.random()
        if step < 0.05:
            qm.force_enqueue()
        elif step < 0.1 and qm.containers[3].prepare:
            taken += len(qm.containers[3].pop().lines_list)    # past the manager
        while rng.random() < 0.4:
            earliest = min(c.min_index for c in qm.containers)
            batch = qm.get()
            assert (batch is None) == (qm.ready() == 0 and earliest > 400)
            if batch is None:
                break
            assert batch.lines_list[0].num_line == earliest
            taken += len(batch.lines_list)
    qm.merge_rest()
    firsts = []
    while (batch := qm.get()) is not None:
        firsts.append(batch.lines_list[0].num_line)
        taken += len(batch.lines_list)
    assert firsts == sorted(firsts) and taken == 400 and qm.ready() == 0


def test_length_above_the_last_edge_is_refused():
    with pytest.raises(ValueError):
        Bt.QueueManager([0, 8], batchsize=2).put(line(0, 9))


def test_a_copy_is_a_manager_of_its_own():
    qm = Bt.QueueManager([2, 8, 40], batchsize=2)
    qm.put(line(0, 5))
    twin = copy.deepcopy(qm)
    twin.put(line(1, 5))
    assert qm.get() is None and [l.num_line for l in twin.get().lines_list] == [0, 1]
