"""Bit identity of a pooled-only call with the full pass on both sides of the row counts at which the plans change their costs (257, 1536, 2400 and 4096 rows),
and between them where float32 launches take tiles whose four waves share K."""
import pytest

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")

import test_gpu_same_bits as bits  # noqa: E402
from test_gpu_same_bits import dirs as dirs, models as models, pb as pb  # noqa: E402,F401


@pytest.mark.parametrize("B,S", [(2, 128), (1, 257), (5, 128), (11, 128), (12, 128), (13, 119), (16, 150), (17, 142), (32, 128), (33, 125), (30, 200)])
@pytest.mark.parametrize("size,precision", bits.SIZES)
def test_first_tokens_alone(pb, models, size, precision, B, S):  # noqa: F811
    bits.test_pooled_only_call_has_the_bits_of_the_full_pass(pb, models, size, precision, B, S)
