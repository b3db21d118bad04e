"""A bucket without a manager keeps nothing of the batches that were taken from it."""
import numpy as np
import pytest

from cudabert_amd import batching as Bt


def line(num):
    return Bt.TaggedLine(num, None, np.ones(4), np.ones(4), np.zeros(4))


@pytest.mark.parametrize("batchsize", [1, 3])
def test_nothing_stays(batchsize):
    bucket = Bt.BatchContainer(0, 8, batchsize)
    for num in range(60):
        bucket.put(line(num))
        while bucket.prepare:
            bucket.pop()
    bucket.force_enqueue()
    assert not bucket.temp and not bucket.prepare and not bucket.queue
