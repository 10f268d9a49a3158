"""A step's embedding rows and first norm in one launch, against the two of them.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


@pytest.mark.parametrize("dim", [8, 768, 2048, 2056, 8192])
@pytest.mark.parametrize("shape", [(1, 1), (3, 5), (513,)])
def test_rows(dim, shape):
    from magicdec_amd import ops
    g = torch.Generator().manual_seed(dim)
    table, w = torch.randn(100, dim, generator=g).to(BF).to(DEV), torch.randn(dim, generator=g).to(BF).to(DEV)
    wide = torch.randint(0, 100, (*shape, 2), generator=g).to(DEV)
    for ids in (wide[..., 0].contiguous(), wide[..., 1]):                       # dense and strided
        x, y = ops.embed_rmsnorm(ids, table, w, 1e-5)
        want = torch.nn.functional.embedding(ids.reshape(-1), table)
        assert torch.equal(x, want) and torch.equal(y, ops.rmsnorm(want, w, 1e-5))


def test_outside():
    from magicdec_amd import ops
    table, w = torch.ones(4, 64, dtype=BF, device=DEV), torch.ones(64, dtype=BF, device=DEV)
    x, y = ops.embed_rmsnorm(torch.tensor([-1, 3, 4, 1 << 40], device=DEV), table, w, 1e-5)
    assert [bool(r.isnan().all()) for r in x] == [True, False, True, True] == [bool(r.isnan().all()) for r in y]
    ids = torch.zeros(2, dtype=torch.int64, device=DEV)
    for bad in ((ids.int(), table, w), (ids.cpu(), table, w), (ids, table.float(), w), (ids, table[:, ::2], w[::2]), (ids, table, w[:32]),
                (ids[:0], table, w), (ids, table[:, :60].contiguous(), w[:60])):
        assert not ops.embed_rmsnorm_supported(*bad)
        with pytest.raises(ValueError):
            ops.embed_rmsnorm(*bad, 1e-5)
