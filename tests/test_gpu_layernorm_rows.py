"""The row kernels of LayerNorm give a row the same bits whichever of them a launch of its size takes, and the copy for the
next GEMM is the result exactly (split) or rounded once (packed).  Rows on both sides of the lines at which the kernel changes."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
PACKED, NO_RESIDUAL, SPLIT = 4, 16, 64


def layernorm(x, y, g, b, layout, flags=0):
    """(result, GEMM-operand copy) of cubert_op_add_layernorm; y is [parts, rows, H]."""
    from cudabert_amd import pybert
    lib = pybert.lib
    lib.cubert_split_bytes.argtypes, lib.cubert_split_bytes.restype = [ctypes.c_size_t] * 2, ctypes.c_size_t
    parts, rows, H = y.shape
    x = x.clone()
    n = lib.cubert_split_bytes(rows, H) if layout == SPLIT else lib.cubert_packed_bytes(rows, H * 2)
    xb = torch.full((n,), 0x5a, dtype=torch.uint8, device="cuda")
    pybert.check(lib.cubert_op_add_layernorm(x.data_ptr(), y.data_ptr(), 0, g.data_ptr(), b.data_ptr(), xb.data_ptr(), rows, H,
                                             layout | flags | (parts << 8 if parts > 1 else 0), None))
    torch.cuda.synchronize()
    return x, xb


def operands(rows, H, parts):
    gen = torch.Generator().manual_seed(rows + H)
    return [t.cuda() for t in (torch.randn(rows, H, generator=gen), torch.randn(parts, rows, H, generator=gen) + 3.0,
                               torch.randn(H, generator=gen), torch.randn(H, generator=gen))]


def reference(x, y, g, b, add_x):
    d = y.double().sum(0) + (x.double() if add_x else 0.0)
    return (d - d.mean(1, keepdim=True)) / torch.sqrt(d.var(1, unbiased=False, keepdim=True) + 1e-12) * g.double() + b.double()


@pytest.mark.parametrize("H", [32, 160, 768, 1024])
@pytest.mark.parametrize("rows,layout", [(1, SPLIT), (800, SPLIT), (801, SPLIT), (807, SPLIT), (1000, SPLIT),
                                         (1, PACKED), (4096, PACKED), (4097, PACKED)])
@pytest.mark.parametrize("flags", [0, NO_RESIDUAL])
def test_rows_do_not_depend_on_the_launch_size(H, rows, layout, flags):
    x, y, g, b = operands(rows, H, 1)
    out, xb = layernorm(x, y, g, b, layout, flags)
    # statistics and normalisation: a few dozen float32 roundings of values of a few units
    assert float((out.double() - reference(x, y, g, b, flags == 0)).abs().max()) < 4e-6 * (1 + float(g.abs().max())) * 4
    cut = max(1, rows // 2 if rows <= 1600 else 700)         # the last rows in a short launch of their own
    tail, _ = layernorm(x[-cut:].contiguous(), y[:, -cut:].contiguous(), g, b, layout, flags)
    assert torch.equal(out[-cut:], tail)
    if layout == SPLIT:
        u = xb.view(torch.bfloat16).view(-1, H // 16, 3, 2, 32, 8).double().sum(2).permute(0, 3, 1, 2, 4).reshape(-1, H)
        assert torch.equal(u[:rows], out.double())
        if rows % 32:                                        # the padding rows of the last block are left alone
            pad = xb.view(-1, H // 16, 3, 2, 32, 16)[-1].permute(3, 0, 1, 2, 4)[rows % 32:]
            assert (pad == 0x5a).all()
    else:
        from cudabert_amd import pybert
        idx = np.array([[pybert.lib.cubert_packed_offset(r, 2 * c, 2 * H) // 2 for c in range(H)] for r in (0, rows // 2, rows - 1)])
        got = xb.view(torch.bfloat16)[torch.from_numpy(idx).cuda()]
        assert torch.equal(got, out[[0, rows // 2, rows - 1]].bfloat16())


@pytest.mark.parametrize("parts", [2, 3, 4, 5, 9, 16])
@pytest.mark.parametrize("rows,H,layout", [(1, 32, SPLIT), (77, 768, PACKED), (130, 1024, SPLIT)])
def test_partial_sums(parts, rows, H, layout):
    x, y, g, b = operands(rows, H, parts)
    out, _ = layernorm(x, y, g, b, layout)
    summed = y[0].clone()
    for p in range(1, parts):
        summed += y[p]
    whole, _ = layernorm(x, summed[None].contiguous(), g, b, layout)
    assert torch.equal(out, whole)
    assert float((out.double() - reference(x, y, g, b, True)).abs().max()) < 1e-4
