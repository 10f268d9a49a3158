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


@pytest.mark.parametrize("graphs", [False, True])
def test_an_id_outside_the_table_stays_in_its_request(graphs):
    """The fixed-batch engines look no ids up on the host: one outside the table leaves its own request without numbers (token 0) and
    the others as they are, in a prompt and in a step."""
    from magicdec_amd.Engine.model_core import transformer_configs
    from magicdec_amd.Engine.SnapKV.backend import LMBackend
    transformer_configs["embed-test"] = dict(block_size=512, n_layer=2, n_head=2, n_local_heads=1, dim=128, intermediate_size=256, vocab_size=64)
    g = torch.Generator().manual_seed(0)
    ids, step = torch.randint(4, 64, (3, 150), generator=g), torch.randint(4, 64, (3, 1), generator=g)
    seen = []
    for bad in (None, 64, -3):
        e = LMBackend(dtype=BF, device=DEV)
        e.load_model("none/embed-test/model.pth", use_tp=False)
        if graphs:
            e.compile()
        e.setup_caches(max_batch_size=3, max_seq_length=256)
        prompt, one = ids.clone(), step.clone()
        if bad is not None:
            prompt[1, 70] = bad
        tokens, logits = e.encode(prompt.to(DEV)), e.model._last_logits.view(3, 22, -1).clone()
        if bad is not None:
            one[1] = bad
        for _ in range(2):
            nxt = e.inference(one.to(DEV), benchmark=True)
        seen.append((tokens, logits, nxt))
    for tokens, logits, nxt in seen[1:]:
        assert logits[1].isnan().all() and not tokens[1].any() and int(nxt[1]) == 0
        for b in (0, 2):
            assert torch.equal(logits[b], seen[0][1][b]) and torch.equal(tokens[b], seen[0][0][b]) and torch.equal(nxt[b], seen[0][2][b])
