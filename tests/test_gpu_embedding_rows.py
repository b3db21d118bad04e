"""Embedding + LayerNorm of few rows (a workgroup per row) against float64, and against the kernel with a wave per row, which the
same lines repeated to more than 4096 rows take: the same bits in float32 result, mask row and GEMM-operand copy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# |x| < 6, as in test_gpu_layernorm_slots.py: about 10 roundings of 6e-8 relative to 6, 1 / sigma a few more; gamma up to 1.5
ATOL = 1e-5


@pytest.mark.parametrize("H", [4, 124, 128, 132, 256, 260, 768, 1020, 1024])
@pytest.mark.parametrize("B,S", [(1, 1), (1, 17), (3, 33), (2, 64)])
@pytest.mark.parametrize("masked", [False, True])
def test_few_rows(H, B, S, masked):
    from cudabert_amd import pybert as pb
    V, Sp, times = 50, (S + 31) // 32 * 32, 4096 // (B * S) + 1
    g = torch.Generator().manual_seed(H + S)
    word, pos, typ = (torch.randn(n, H, generator=g) for n in (V, S, 2))
    gamma, beta = torch.rand(H, generator=g) + 0.5, torch.randn(H, generator=g)
    ids = torch.randint(0, V, (B, S), generator=g, dtype=torch.int32)
    ids[0, 0], ids[-1, -1] = V + 3, -1                      # out of the vocabulary: clamped
    seg = torch.randint(0, 2, (B, S), generator=g, dtype=torch.int32)
    mask = torch.randint(0, 2, (B, S), generator=g, dtype=torch.int32)
    table = [t.cuda() for t in (word, pos, typ, gamma, beta)]

    def run(n):
        io = [t.repeat(n, 1).cuda() for t in (ids, seg, mask)]
        x = torch.full((n * B * S + 2, H), 7.0, device="cuda")
        xb = torch.zeros(n * B * S, H, dtype=torch.bfloat16, device="cuda")
        m = torch.full((n * B, Sp), 7.0, device="cuda")
        pb.check(pb.lib.cubert_op_embed_layernorm(io[0].data_ptr(), io[1].data_ptr(), io[2].data_ptr() if masked else None,
                                                  *[t.data_ptr() for t in table], x.data_ptr(), xb.data_ptr(), m.data_ptr(),
                                                  n * B, S, H, V, 2, 0, torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert (x[n * B * S:] == 7.0).all()
        return x[:B * S].cpu(), xb[:B * S].cpu(), m[:B].cpu()

    x, xb, m = run(1)
    e = ((word[ids.clamp(0, V - 1).long()] + pos) + typ[seg.long()]).reshape(B * S, H).double().numpy()
    want = (e - e.mean(1, keepdims=True)) / np.sqrt(e.var(1, keepdims=True) + 1e-12) * gamma.double().numpy() + beta.double().numpy()
    if H > 4:                                               # (four features: sigma may be small against the values)
        np.testing.assert_allclose(x.double().numpy(), want, rtol=0, atol=ATOL)
    assert torch.equal(m[:, :S], (1.0 - mask.float()) * -10000.0 if masked else torch.zeros(B, S))
    assert torch.isneginf(m[:, S:]).all()
    for a, b in zip((x, xb, m), run(times)):
        assert torch.equal(a, b)
