"""LayerNorm GEMMs on both sides of the row counts where the launcher's own choice of the tile changes, for the widths whose bands
are one to three workgroups: whatever it takes has the bits of every tile asked for by name."""
import pytest

from test_gpu_layernorm_rows192 import launch

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("N,M", [(768, 10240), (768, 10241), (768, 15360), (768, 15361), (768, 20481), (512, 16384), (512, 16385),
                                 (512, 24577), (256, 32769), (256, 49153)])
def test_the_choice_is_among_equals(N, M):
    from cudabert_amd import pybert as pb
    K, flags = 128, pb.X_PACKED | pb.W_PACKED | pb.Y_PACKED
    g = torch.Generator().manual_seed(M)
    X = torch.randn(pb.lib.cubert_packed_bytes(M, K * 2) // 2, generator=g).to(torch.bfloat16).cuda()
    W = (torch.randn(pb.lib.cubert_packed_bytes(N, K * 2) // 2, generator=g) * 0.05).to(torch.bfloat16).cuda()
    vec = [torch.randn(N, generator=g).cuda() for _ in range(3)]
    R = torch.randn(M, N, generator=g).cuda()
    out = []
    for tile in (0, 384, 386, 256):
        Y = torch.zeros(M, N, device="cuda")
        xb = torch.zeros(pb.lib.cubert_packed_bytes(M, N * 2) // 2, dtype=torch.int16, device="cuda")
        pb.check(launch(pb, X, W, vec, R, Y, xb, M, N, K, tile, flags))
        out.append((Y, xb))
    assert torch.isfinite(out[0][0]).all()
    for Y, xb in out[1:]:
        assert torch.equal(Y, out[0][0]) and torch.equal(xb, out[0][1])
