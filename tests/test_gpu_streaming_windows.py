"""Several portions of a prompt through the StreamingLLM cache at once, against one after the other.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SINK = 16


@pytest.mark.parametrize("KH,D,portion", [(1, 16, 128), (8, 64, 128), (5, 128, 128), (2, 64, 7)])
@pytest.mark.parametrize("kv_len", [130, 256, 257, 300, 513])
@pytest.mark.parametrize("held,tokens", [(0, 129), (0, 384), (1, 250), (1, 1000), (2, 500), (9, 131), (9, 900)])
def test_windows(KH, D, portion, kv_len, held, tokens):
    """Bit for bit what portions shifted in, appended and rotated one by one leave: every window, and the cache behind them."""
    from magicdec_amd import ops
    B, ppr, g = 3, kv_len // 128 + 1, torch.Generator().manual_seed(kv_len + tokens + held)
    ctx = min(held * portion, kv_len)
    table = ops.RopeTable(1024, D, 10000.0, 1.0, device=DEV)
    cache = torch.randn(B * ppr, 2, 128, KH, D, generator=g).bfloat16().to(DEV)
    new = torch.randn(B, tokens, 2 * KH + 1, D, generator=g).bfloat16().to(DEV)
    flat = new.view(B * tokens, 2 * KH + 1, D)
    C = -(-tokens // portion)
    for turn in (False, True):
        windows = torch.full((B * C * ppr, 2, 128, KH, D), 7.0, dtype=torch.bfloat16, device=DEV)
        following = torch.empty_like(cache)
        ops.streaming_windows(flat[:, :KH], flat[:, KH:2 * KH], cache, windows, following, portion, ctx, kv_len, SINK, ppr, table, turn)
        one, at = cache.clone(), ctx
        for c in range(C):
            part = new[:, c * portion:(c + 1) * portion]
            n = part.shape[1]
            rows = part.reshape(B * n, 2 * KH + 1, D)
            if at + n <= kv_len:
                view = one.view(B, ppr, 2, 128, KH, D).transpose(1, 2).reshape(B, 2, ppr * 128, KH, D)
                for j in (0, 1):
                    view[:, j, at:at + n] = part[:, :, j * KH:(j + 1) * KH]
                one = view.view(B, 2, ppr, 128, KH, D).transpose(1, 2).reshape(cache.shape).contiguous()
                valid = at + n
            else:
                ops.streaming_shift_append(rows[:, :KH], rows[:, KH:2 * KH], one, n, kv_len, SINK, ppr)
                valid = kv_len
            at = min(at + n, kv_len)
            want = torch.empty_like(one)
            ops.streaming_rotate(one, want, B, valid, ppr, table)
            got = windows.view(B, C, ppr, 2, 128, KH, D)[:, c].transpose(1, 2).reshape(B, 2, ppr * 128, KH, D)
            want = want.view(B, ppr, 2, 128, KH, D).transpose(1, 2).reshape(got.shape)
            assert torch.equal(got[:, :, :valid], want[:, :, :valid])
            assert torch.all(got[:, :, valid:] == 7.0)
        if turn:
            ops.streaming_rotate(one, one, B, valid, ppr, table)
        assert torch.equal(following, one)


def test_what_it_does_not_take():
    from magicdec_amd import ops
    table = ops.RopeTable(512, 64, 10000.0, 1.0, device=DEV)
    cache = torch.zeros(4, 2, 128, 2, 64, dtype=torch.bfloat16, device=DEV)
    new, windows = torch.zeros(2 * 200, 2, 64, dtype=torch.bfloat16, device=DEV), torch.zeros(8, 2, 128, 2, 64, dtype=torch.bfloat16, device=DEV)
    good = (new, new, cache, windows, torch.empty_like(cache), 128, 0, 200, SINK, 2, table, False)
    ops.streaming_windows(*good)
    for at, bad in ((0, new.float()), (0, new[:, :1]), (2, cache[:, :, :64]), (3, windows[:4]), (4, cache[:2]), (4, cache), (5, 0), (6, 201),
                    (7, 300), (7, 16)):
        args = list(good)
        args[at] = bad
        with pytest.raises((ValueError, RuntimeError)):
            ops.streaming_windows(*args)


@pytest.mark.parametrize("which", ["draft", "self"])
@pytest.mark.parametrize("budget,batch,prompt", [(257, 2, 130), (257, 3, 384), (257, 1, 900), (200, 4, 1500), (513, 2, 1024), (129, 33, 600)])
def test_engines(which, budget, batch, prompt, monkeypatch):
    """Prompts in one pass and chunk by chunk: tables and lengths equal; rows, logits and the step behind them those of 16-bit arithmetic."""
    import magicdec_amd.Engine.backend_core as core
    from magicdec_amd.Engine.model_core import transformer_configs
    transformer_configs["windows-test"] = dict(block_size=4096, n_layer=2, n_head=8, n_local_heads=2, dim=512, intermediate_size=1024,
                                               vocab_size=512)
    ids = torch.randint(4, 512, (batch, prompt), generator=torch.Generator().manual_seed(prompt)).to(DEV)
    seen = []
    for rows in (core.PROMPT_ROWS, 0):
        monkeypatch.setattr(core, "PROMPT_ROWS", rows)
        if which == "draft":
            from magicdec_amd.Engine.StreamingLLM.backend_draft import LMBackend_Draft
            e = LMBackend_Draft(dtype=torch.bfloat16, device=DEV)
            e.load_model("none/windows-test/model.pth", use_tp=False)
            e.setup_caches(max_batch_size=batch, draft_budget=budget)
            run, name, lens, state, step = e.encode, "kv_cache", "cachelens", e._t, e.inference
        else:
            from magicdec_amd.Engine.StreamingLLM.backend import LMBackend
            e = LMBackend(dtype=torch.bfloat16, device=DEV, dec_len=4)
            e.load_model("none/windows-test/model.pth", use_tp=False)
            e.setup_caches(max_batch_size=batch, max_seq_length=2048, draft_budget=budget)
            e.clear_kv()
            run, name, lens, state, step = e.draft_encode, "draft_cache", "draft_cachelens", e._d, e.speculate
        tokens = run(ids)
        logits, tab = e.model._last_logits.float(), state.table()
        kept = [getattr(b.attention.kv_cache, name).float().clone() for b in e.model.layers]
        seen.append(dict(tokens=tokens, lens=getattr(e, lens).clone(), tab=[t.clone() for t in (tab.indices, tab.indptr, tab.last_page_len)],
                         close=[logits, *kept]))
        step(ids[:, :1])
        seen[-1]["close"].append(e.model._last_logits.float())
    a, b = seen
    assert a["tokens"].shape == b["tokens"].shape == (batch, (prompt - 1) % 128 + 1)
    assert torch.equal(a["lens"], b["lens"]) and all(torch.equal(x, y) for x, y in zip(a["tab"], b["tab"]))
    for x, y in zip(a["close"], b["close"]):                          # each within 0.8 % of exact arithmetic
        assert (x - y).norm() <= 0.016 * y.norm()
