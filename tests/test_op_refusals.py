"""Calls of the op entry points that the launchers have to refuse on the host: each asks for a kernel form that would write or
read past its buffers.  The operands are addresses that nothing may touch; no GPU is needed, the refusal comes first."""
import pytest

BF16, F32, SPLIT = 1, 0, 2
X_UNITS, W_UNITS, Y_UNITS = 1 | 128, 2 | 1 << 24, 4 | 1 << 25      # each with its _PACKED flag
SKINNY12, SKINNY22 = 97, 98
A = 1 << 20                                                          # 16-byte aligned, never dereferenced


@pytest.fixture(scope="module")
def pb():
    from cudabert_amd import pybert
    return pybert


def refused(pb, match, rc):
    assert rc != 0
    with pytest.raises(pb.CubertError, match=match):
        pb.check(rc)


@pytest.mark.parametrize("tile", [SKINNY12, SKINNY22])
@pytest.mark.parametrize("epilogue,out,flags", [
    (1, F32, X_UNITS | W_UNITS),                 # GELU, float32 rows: the kernel writes bf16 units, past such a Y
    (0, BF16, X_UNITS | W_UNITS),                # plain bias in bf16
    (1, BF16, X_UNITS | W_UNITS | 4),            # GELU in the packed layout
    (2, F32, X_UNITS | W_UNITS),                 # tanh
    (0, F32, 1 | W_UNITS),                       # an operand in the packed layout
])
def test_skinny_tile_takes_only_what_its_kernel_writes(pb, tile, epilogue, out, flags):
    refused(pb, "skinny", pb.lib.cubert_op_gemm(A, A, A, A, 1, 4096, 1024, 1024, BF16, out, epilogue, tile, flags, None))


@pytest.mark.parametrize("partition", [1, 3, 5, 9, 14])
@pytest.mark.parametrize("elt", [BF16, F32, SPLIT])
def test_xcd_partition_is_checked_for_every_operand_type(pb, elt, partition):
    """tile_of_block divides by the partition and takes block rows from it: another value leaves tiles out and reads past X."""
    flags = (partition + 1) << 16
    refused(pb, "XCD partition", pb.lib.cubert_op_gemm(A, A, A, A, 256, 256, 256, 256, elt, F32, 0, 128, flags, None))
    refused(pb, "XCD partition", pb.lib.cubert_op_gemm_qkv(A, A, A, A, A, A, 2, 128, 4, elt, 128, flags, None))
