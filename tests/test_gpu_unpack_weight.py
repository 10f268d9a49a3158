"""The streaming weight layout back into rows, at the ends of its tiles.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [16, 80, 512, 528, 2064])
@pytest.mark.parametrize("N", [2, 30, 32, 34, 96, 1030])
@pytest.mark.parametrize("halves", [False, True])
def test_unpack(N, K, halves):
    from magicdec_amd import ops
    w = torch.randn(N, K, generator=torch.Generator().manual_seed(N + K)).bfloat16().cuda()
    assert torch.equal(ops.PackedWeight(w, swiglu=halves).unpack(), w)
