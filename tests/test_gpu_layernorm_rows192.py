"""The 256 features x 192 tokens GEMM with LayerNorm in its epilogue: tiles of 192 rows whose groups of 64 lie in one or two of
the packed layout's blocks of 256, waves of 96 rows, ragged last tiles.  K is summed in the order of the 256 x 256 kernel and the
statistics by one recipe, so float32 result and bf16 copy equal that kernel's bit for bit (which test_gpu_ops.py holds against
float64 and against the row kernel)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
T192, T256 = 386, 256


def launch(pb, X, W, vec, R, Y, xb, M, N, K, tile, flags):
    ws = torch.zeros(pb.lib.cubert_gemm_layernorm_workspace_bytes(M) // 4, dtype=torch.int32, device="cuda")
    rc = pb.lib.cubert_op_gemm_residual_layernorm(X.data_ptr(), W.data_ptr(), vec[0].data_ptr(), R.data_ptr(), vec[1].data_ptr(),
                                                  vec[2].data_ptr(), Y.data_ptr(), xb.data_ptr(), ws.data_ptr(), M, N, K, K, tile, flags,
                                                  torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert not ws[:64 + 2 * 16384].any()                  # nobody gave up, counters back at zero
    return rc


@pytest.mark.parametrize("N,K", [(256, 128), (768, 768), (1024, 1024), (1024, 4096)])
@pytest.mark.parametrize("M", [1, 31, 95, 97, 191, 192, 193, 257, 500, 769, 4607])
@pytest.mark.parametrize("form", ["rowmajor", "packed", "units"])
def test_same_bits_as_the_256_tile(M, N, K, form):
    from cudabert_amd import pybert as pb
    g = torch.Generator().manual_seed(M + N + K)
    nx, nw = pb.lib.cubert_packed_bytes(M, K * 2) // 2, pb.lib.cubert_packed_bytes(N, K * 2) // 2
    # (in a packed layout any values are a matrix: both kernels read the same one)
    X = torch.randn(M * K if form == "rowmajor" else nx, generator=g).to(torch.bfloat16).cuda()
    W = (torch.randn(N * K if form == "rowmajor" else nw, generator=g) * 0.05).to(torch.bfloat16).cuda()
    vec = [torch.randn(N, generator=g).cuda() for _ in range(3)]
    R = torch.randn(M, N, generator=g).cuda()
    flags = {"rowmajor": 0, "packed": pb.X_PACKED | pb.W_PACKED | pb.Y_PACKED,
             "units": pb.X_PACKED | pb.W_PACKED | pb.Y_PACKED | 128 | 1 << 24}[form]
    out = []
    for tile in (T192, T256):
        Y = torch.full((M + 2, N), 7.0, device="cuda")
        xb = torch.full((pb.lib.cubert_packed_bytes(M, N * 2) // 2,), 0x7fc0, dtype=torch.int16, device="cuda")
        if tile == T192:
            Y[1:M + 1].copy_(R)                           # in place on the residual, as the model runs it
        pb.check(launch(pb, X, W, vec, Y[1:] if tile == T192 else R, Y[1:], xb, M, N, K, tile, flags))
        out.append((Y.cpu().numpy(), xb.cpu().numpy()))
    assert np.isfinite(out[0][0]).all()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("M", [8192, 8193, 12288, 12289])
def test_the_launcher_chooses_among_equals(M):
    """Around the row counts where the launcher's own choice of the tile changes (N = 1024): the same bits."""
    from cudabert_amd import pybert as pb
    N, K, flags = 1024, 128, pb.X_PACKED | pb.W_PACKED | pb.Y_PACKED
    g = torch.Generator().manual_seed(M)
    X = torch.randn(pb.lib.cubert_packed_bytes(M, K * 2) // 2, generator=g).to(torch.bfloat16).cuda()
    W = (torch.randn(pb.lib.cubert_packed_bytes(N, K * 2) // 2, generator=g) * 0.05).to(torch.bfloat16).cuda()
    vec = [torch.randn(N, generator=g).cuda() for _ in range(3)]
    R = torch.randn(M, N, generator=g).cuda()
    out = []
    for tile in (0, T192, T256):
        Y = torch.zeros(M, N, device="cuda")
        xb = torch.zeros(pb.lib.cubert_packed_bytes(M, N * 2) // 2, dtype=torch.int16, device="cuda")
        pb.check(launch(pb, X, W, vec, R, Y, xb, M, N, K, tile, flags))
        out.append((Y, xb))
    for Y, xb in out[1:]:
        assert torch.equal(Y, out[0][0]) and torch.equal(xb, out[0][1])


def test_refusals():
    from cudabert_amd import pybert as pb
    z = torch.zeros(1 << 20, device="cuda")
    # K not a multiple of 128; a plain GEMM
    assert launch(pb, z, z, [z, z, z], z, z, z, 256, 256, 160, T192, 0) != 0
    assert pb.lib.cubert_op_gemm(z.data_ptr(), z.data_ptr(), z.data_ptr(), z.data_ptr(), 256, 256, 256, 256, 1, 0, 0, T192, 0, None) != 0
