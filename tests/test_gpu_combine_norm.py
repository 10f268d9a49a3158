"""The combine + residual + norm launch where a row's vectors go to one, two and four groups of threads: bit for bit the three launches.
On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


@pytest.mark.parametrize("N", [8, 2040, 2048, 2056, 4088, 4096, 4104, 5120, 8184, 8192])
@pytest.mark.parametrize("M,K", [(1, 1408), (33, 2304)])
@pytest.mark.parametrize("bias", [False, True])
def test_combine(M, N, K, bias):
    from magicdec_amd import ops
    g = torch.Generator().manual_seed(M + N)
    x, r = torch.randn(M, K, generator=g).to(BF).to(DEV), torch.randn(M, N, generator=g).to(BF).to(DEV)
    w, nw = ops.PackedWeight((torch.randn(N, K, generator=g) * 0.05).to(BF).to(DEV)), torch.randn(N, generator=g).to(BF).to(DEV)
    b, ws = torch.randn(N, generator=g).to(BF).to(DEV) if bias else None, ops.AttnWorkspace(DEV)
    assert ops.linear_add_rmsnorm_supported(M, N, K)
    h, y = ops.linear_add_rmsnorm(x, w, r, nw, 1e-5, b, workspace=ws)
    h1, y1 = ops.add_rmsnorm(r, ops.linear(x, w, b, workspace=ws), nw, 1e-5)
    assert torch.equal(h, h1) and torch.equal(y, y1)
