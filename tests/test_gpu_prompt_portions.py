"""A prompt in longer portions against portions of 128 tokens: the same tables, lengths and fp8 scales, the rows and logits of 16-bit
arithmetic.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def engine(which, kv, batch, limit):
    from magicdec_amd.Engine.model_core import transformer_configs
    transformer_configs["portions-test"] = dict(block_size=4096, n_layer=2, n_head=8, n_local_heads=2, dim=512, intermediate_size=1024,
                                                vocab_size=512)
    if which == "draft":
        from magicdec_amd.Engine.SnapKV.backend_draft import LMBackend_Draft
        e, kw = LMBackend_Draft(dtype=torch.bfloat16, device=DEV, draft_budget=129), dict(draft_budget=129, window_size=32)
    elif which == "spec":
        from magicdec_amd.Engine.SnapKV.backend import LMBackend
        e, kw = LMBackend(dtype=torch.bfloat16, device=DEV, dec_len=4, draft_dec_len=1), dict(draft_budget=129, window_size=32, kv_dtype=kv)
    elif which == "stream":
        from magicdec_amd.Engine.StreamingLLM.backend import LMBackend
        e, kw = LMBackend(dtype=torch.bfloat16, device=DEV, dec_len=4), dict(draft_budget=129, kv_dtype=kv)
    else:
        from magicdec_amd.Engine.SnapKV.backend import LMBackend
        e, kw = LMBackend(dtype=torch.bfloat16, device=DEV, dec_len=4), dict(kv_dtype=kv)
    e.load_model("none/portions-test/model.pth", use_tp=False)
    e.setup_caches(max_batch_size=batch, max_seq_length=limit, **kw)
    return e


@pytest.mark.parametrize("which,kv,batch,prompt", [
    ("plain", "bf16", 3, 1), ("plain", "bf16", 1, 128), ("plain", "bf16", 2, 129), ("plain", "bf16", 3, 256), ("plain", "bf16", 5, 1337),
    ("plain", "bf16", 33, 700), ("plain", "bf16", 65, 300), ("plain", "fp8", 2, 128), ("plain", "fp8", 2, 200), ("plain", "fp8", 3, 1500),
    ("spec", "bf16", 2, 1056), ("spec", "fp8", 3, 416), ("draft", "bf16", 4, 800), ("stream", "bf16", 2, 555), ("stream", "fp8", 2, 1024)])
def test_longer_portions(which, kv, batch, prompt, monkeypatch):
    import magicdec_amd.Engine.backend_core as core
    ids = torch.randint(4, 512, (batch, prompt), generator=torch.Generator().manual_seed(prompt)).to(DEV)
    seen = []
    for rows in (core.PROMPT_ROWS, 0):
        monkeypatch.setattr(core, "PROMPT_ROWS", rows)
        e = engine(which, kv, batch, 2048)
        parts = e._portions(prompt)
        # in order and whole, each at a page's start
        assert [a for a, _ in parts] == [0] + [a + n for a, n in parts[:-1]] and sum(parts[-1]) == prompt
        assert all(a % 128 == 0 for a, _ in parts) and all(n * batch <= max(rows, 128 * batch) for _, n in parts)
        assert rows == 0 or kv != "fp8" or parts[0][1] <= 128
        for _ in range(2):                                           # (a second prompt over the first one's state)
            tokens = e.encode(ids)
        kvs = [b.attention.kv_cache for b in e.model.layers]
        seen.append(dict(tokens=tokens, logits=e.model._last_logits.float(), lens=e.cachelens, pages=e._t.table(),
                         scales=[s for c in kvs for s in (c.scales() or ())],
                         kept=[c.draft_cache.float() for c in kvs] if which in ("spec", "draft") else [], rows=[c.kv_cache.float() for c in kvs]))
    a, b = seen
    assert a["tokens"].shape == b["tokens"].shape == (batch, (prompt - 1) % 128 + 1)
    assert torch.equal(a["lens"], b["lens"]) and a["pages"].max_pages == b["pages"].max_pages
    assert all(torch.equal(getattr(a["pages"], k), getattr(b["pages"], k)) for k in ("indices", "indptr", "last_page_len"))
    assert all(torch.equal(x, y) for x, y in zip(a["scales"], b["scales"]))
    # each within 0.8 % of exact arithmetic; an fp8 row rounds to 2^-4 of itself, so a moved rounding shows as far as that in few places
    for x, y in zip([a["logits"]] + a["rows"], [b["logits"]] + b["rows"]):
        rel = 0.016 if kv == "bf16" else 0.03
        assert (x - y).norm() <= rel * y.norm()
        # ... and no shift that the rows share: independent differences of that size leave rel / sqrt(n) along y
        x, y = x.double(), y.double()
        assert abs(((x - y) * y).sum()) <= 6 * rel * (y * y).sum() / y.count_nonzero() ** 0.5
    # the select over the same window: but for scores on the edge, the same rows
    for x, y in zip(a["kept"], b["kept"]):
        near = (x - y).norm(dim=-1) <= 0.05 * y.norm(dim=-1)
        assert near.double().mean() > 0.8


@pytest.mark.parametrize("which,batch,prompt", [("spec", 2, 1440), ("draft", 4, 2080), ("spec", 1, 3104)])
def test_longer_portions_behind_split_keys(which, batch, prompt, monkeypatch):
    """Where a chunk's keys are split over workgroups the chunks' roundings are independent of the portions' from the first layer's
    attention on: the same bounds on rows and logits as above.  Of the rows kept for the draft, the first layer's are of the same scores but
    for the products' rounding; behind it the scores, as close as random weights make them, move by 1 % (0.70 to 0.85 of the rows stay,
    0.78 to 0.97 where two orders of whole keys round partly alike)."""
    import magicdec_amd.Engine.backend_core as core
    ids = torch.randint(4, 512, (batch, prompt), generator=torch.Generator().manual_seed(prompt)).to(DEV)
    seen = []
    for rows in (core.PROMPT_ROWS, 0):
        monkeypatch.setattr(core, "PROMPT_ROWS", rows)
        e = engine(which, "bf16", batch, 4096)
        e.encode(ids)
        kvs = [b.attention.kv_cache for b in e.model.layers]
        seen.append(([e.model._last_logits.float()] + [c.kv_cache.float() for c in kvs], [c.draft_cache.float() for c in kvs]))
    (a, kept_a), (b, kept_b) = seen
    for x, y in zip(a, b):
        assert (x - y).norm() <= 0.016 * y.norm()
        x, y = x.double(), y.double()
        assert abs(((x - y) * y).sum()) <= 6 * 0.016 * (y * y).sum() / y.count_nonzero() ** 0.5
    for x, y, least in zip(kept_a, kept_b, (0.95, 0.6)):
        assert ((x - y).norm(dim=-1) <= 0.05 * y.norm(dim=-1)).double().mean() > least


@pytest.mark.parametrize("which", ["plain", "draft", "stream_draft"])
def test_portions_where_memory_is_short(which, monkeypatch):
    """With little free memory a prompt runs in single chunks, as it would without longer portions: the same bits."""
    import magicdec_amd.Engine.backend_core as core
    from magicdec_amd.Engine.model_core import transformer_configs
    ids = torch.randint(4, 512, (2, 800), generator=torch.Generator().manual_seed(5)).to(DEV)
    seen = []
    for short in (True, False):
        if which == "stream_draft":
            from magicdec_amd.Engine.StreamingLLM.backend_draft import LMBackend_Draft
            engine("plain", "bf16", 1, 256)                            # (registers the configuration)
            e = LMBackend_Draft(dtype=torch.bfloat16, device=DEV)
            e.load_model("none/portions-test/model.pth", use_tp=False)
            e.setup_caches(max_batch_size=2, draft_budget=257)
        else:
            e = engine(which, "bf16", 2, 1024)
        with monkeypatch.context() as m:
            if short:
                m.setattr(torch.cuda, "mem_get_info", lambda dev=None: (0, 1 << 38))
                m.setattr(torch.cuda, "memory_reserved", lambda dev=None: torch.cuda.memory_allocated(dev) + 3 * 128 * e.model.prompt_row_bytes())
            else:
                m.setattr(core, "PROMPT_ROWS", 0)
            tokens = e.encode(ids)
        kvs = [b.attention.kv_cache for b in e.model.layers]
        seen.append([tokens, e.model._last_logits] + [c.kv_cache for c in kvs] + ([c.draft_cache for c in kvs] if which == "draft" else []))
    assert all(torch.equal(x, y) for x, y in zip(*seen))
