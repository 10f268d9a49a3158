"""The greedy token where a thread's loads end, and among equal maxima.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


@pytest.mark.parametrize("rows,vocab", [(1, 1), (3, 7), (2, 1000), (1, 8192), (2, 8193), (1, 16384), (2, 32767), (3, 32768), (1, 32776), (2, 128256), (1, 16392), (2, 24576), (2, 24584),
                                        (513, 16384)])
@pytest.mark.parametrize("dtype", [BF, torch.float32])
def test_argmax(rows, vocab, dtype):
    from magicdec_amd import ops
    g = torch.Generator().manual_seed(rows + vocab)
    x = torch.randint(-50, 50, (rows, vocab), generator=g).to(dtype).to(DEV)               # many equal maxima: the first one
    assert torch.equal(ops.argmax(x), (x == x.max(-1, keepdim=True).values).int().argmax(-1))
    for at in {0, vocab // 2, vocab - 1}:
        y = x.clone()
        y[:, at] = 60.0
        assert torch.all(ops.argmax(y) == at)
    low = torch.full_like(x, float("-inf"))
    assert torch.all(ops.argmax(low) == 0)
