"""LayerNorm of rows whose last slot of 128 features is full, partly filled or absent, through the kernel with a workgroup per row
(with and without partial sums to add) and the one with a wave per row: against float64, and both kernels the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# |x| < 6: the mean and the deviations are good to about 10 roundings of 6e-8 relative to 6, 1 / sigma to a few more
ATOL = 1e-5


@pytest.mark.parametrize("H", [4, 64, 124, 128, 132, 256, 260, 508, 640, 768, 1020, 1024])
@pytest.mark.parametrize("parts", [1, 2, 4, 5])
def test_slots(H, parts):
    from cudabert_amd import pybert as pb
    from cudabert_amd.pybert import F32
    g = torch.Generator().manual_seed(H + parts)
    rows, many = 37, 4100                                   # above 4096 rows: a wave per row
    y = torch.randn(parts, rows, H, generator=g) / parts ** 0.5
    gamma, beta = torch.rand(H, generator=g) + 0.5, torch.randn(H, generator=g)
    acc = y[0].clone()
    for p in range(1, parts):
        acc += y[p]
    s = acc.double().numpy()
    mean = s.mean(1, keepdims=True)
    want = (s - mean) / np.sqrt(s.var(1, keepdims=True) + 1e-12) * gamma.double().numpy() + beta.double().numpy()
    gd, bd = gamma.cuda(), beta.cuda()

    def run(t, n, k):
        x = torch.zeros(n, H, device="cuda")
        t = t.cuda()
        pb.check(pb.lib.cubert_op_add_layernorm(x.data_ptr(), t.data_ptr(), F32, gd.data_ptr(), bd.data_ptr(), None, n, H,
                                                16 | (k << 8 if k > 1 else 0), torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        return x.cpu()

    got = run(y, rows, parts)
    np.testing.assert_allclose(got.double().numpy(), want, rtol=0, atol=ATOL)
    one = acc.repeat((many + rows - 1) // rows, 1)[:many].contiguous()
    wave = run(one, many, 1)
    assert torch.equal(wave[:rows], run(acc.contiguous(), rows, 1)) and torch.equal(wave[:rows], wave[rows:2 * rows])
    assert torch.equal(wave[:rows], got)
