"""Attention over chunks of keys (bf16, V as rows) at the edges of blocks, chunks and query groups.

The kernel that holds a whole head's K and V^T in LDS (V handed over transposed) does the same arithmetic in the same order, so
the two agree bit for bit; against float64 the bound is that of a bf16 result and bf16 probabilities on values of size up to 4:
2^-9 * 4 for the rounding of the result and as much for those of the probabilities, 1.6e-2 together."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
BF16, V_ROWMAJOR, PER_HEAD = 1, 32, 1 << 20


def masks(S):
    """All keys; a short prefix (later chunks masked whole); nothing but the last key; the middle third; no key at all."""
    m = np.zeros((5, S), np.float32)
    m[0] = 1
    m[1, :max(1, S // 5)] = 1
    m[2, S - 1] = 1
    m[3, S // 3:max(S // 3 + 1, 2 * S // 3)] = 1
    return m


@pytest.mark.parametrize("S", [1, 31, 32, 33, 64, 65, 96, 128, 129, 160, 256, 257, 384, 385, 511, 512])
def test_matches_the_whole_head_kernel_and_float64(S):
    from cudabert_amd import pybert as pb
    mask = masks(S)
    B, heads, Sp = len(mask), 3, (S + 31) // 32 * 32
    gen = torch.Generator().manual_seed(S)
    q, k, v = [torch.randn(B, heads, S, 64, generator=gen).to(torch.bfloat16) for _ in range(3)]
    vt = torch.zeros(B, heads, 64, Sp, dtype=torch.bfloat16)
    vt[..., :S] = v.transpose(2, 3)
    add = torch.full((B, Sp), float("-inf"))
    add[:, :S] = torch.from_numpy((1 - mask) * -10000.0)
    qd, kd, vd, td, md = q.cuda(), k.cuda(), v.cuda(), vt.cuda(), add.cuda()
    rows, whole = [torch.full((B, S, heads, 64), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    pb.check(pb.lib.cubert_op_attention(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), md.data_ptr(), rows.data_ptr(), B, heads, S, 0.125,
                                        BF16, V_ROWMAJOR | PER_HEAD, None))
    pb.check(pb.lib.cubert_op_attention(qd.data_ptr(), kd.data_ptr(), td.data_ptr(), md.data_ptr(), whole.data_ptr(), B, heads, S, 0.125,
                                        BF16, 0, None))
    torch.cuda.synchronize()
    assert torch.equal(rows.view(torch.int16), whole.view(torch.int16))
    sc = q.double() @ k.double().transpose(2, 3) * 0.125 + add[:, None, None, :S].double()
    want = (torch.softmax(sc, -1) @ v.double()).transpose(1, 2)
    err = (rows.cpu().double() - want).abs().amax(dim=(1, 2, 3))
    assert (err[:4] < 1.6e-2).all(), err         # row 4: no visible key, scores near -10000 resolve 1e-3 only
    assert err[4] < 2e-2
