"""The in-place eviction of the StreamingLLM cache where its row groups and column groups end.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("KH,D", [(1, 8), (3, 24), (1, 64), (8, 64), (8, 128)])
@pytest.mark.parametrize("kv_len,n", [(17, 1), (129, 128), (257, 128), (271, 3), (272, 255), (273, 256), (513, 128), (1025, 31), (300, 300)])
def test_shift_append(KH, D, kv_len, n):
    """cache[sink:] = (cache[sink:], new rows)[-(kv_len - sink):], bit for bit, the sink and the rest of the pages untouched."""
    from magicdec_amd import ops
    B, sink, ppr, g = 3, 16, kv_len // 128 + 1, torch.Generator().manual_seed(kv_len + n)
    cache = torch.randn(B * ppr, 2, 128, KH, D, generator=g).bfloat16()
    new = torch.randn(B * n, 2 * KH + 1, D, generator=g).bfloat16()
    rows = cache.view(B, ppr, 2, 128, KH, D).transpose(1, 2).reshape(B, 2, ppr * 128, KH, D).clone()
    for j in (0, 1):
        add = new[:, j * KH:(j + 1) * KH].reshape(B, n, KH, D)
        rows[:, j, sink:kv_len] = torch.cat([rows[:, j, sink:kv_len], add], 1)[:, n:]
    want = rows.view(B, 2, ppr, 128, KH, D).transpose(1, 2).reshape(cache.shape)
    got, dn = cache.to(DEV), new.to(DEV)
    ops.streaming_shift_append(dn[:, :KH], dn[:, KH:2 * KH], got, n, kv_len, sink, ppr)
    assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize("B,KH,D,kv_len,n", [(64, 40, 128, 141, 128), (76, 32, 128, 257, 33), (75, 8, 128, 513, 1), (45, 3, 120, 4999, 1000)])
def test_shift_append_beyond_the_last_level_cache(B, KH, D, kv_len, n):
    """The same where a workgroup moves wider runs, from 266 MB of rows on (the last two: just below), on the device."""
    from magicdec_amd import ops
    sink, ppr, g = 16, kv_len // 128 + 1, torch.Generator(device=DEV).manual_seed(kv_len)
    cache = torch.randn(B * ppr, 2, 128, KH, D, generator=g, device=DEV).bfloat16()
    new = torch.randn(B * n, 2 * KH + 1, D, generator=g, device=DEV).bfloat16()
    rows = cache.view(B, ppr, 2, 128, KH, D).transpose(1, 2).reshape(B, 2, ppr * 128, KH, D).clone()
    for j in (0, 1):
        add = new[:, j * KH:(j + 1) * KH].reshape(B, n, KH, D)
        rows[:, j, sink:kv_len] = torch.cat([rows[:, j, sink:kv_len], add], 1)[:, n:]
    want = rows.view(B, 2, ppr, 128, KH, D).transpose(1, 2).reshape(cache.shape)
    ops.streaming_shift_append(new[:, :KH], new[:, KH:2 * KH], cache, n, kv_len, sink, ppr)
    assert torch.equal(cache, want)
