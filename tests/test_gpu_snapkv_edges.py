"""The SnapKV selection where its column groups, chunks, register accumulators and bins end, against the CPU restatement of the
reference (oracle/magicdec_ref.py).  Queries and keys are small integers: the scores are exact in any order.  On the GPU (-m gpu)."""
import pytest
import torch

from oracle import magicdec_ref as mr

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("page", [128, 48])
@pytest.mark.parametrize("g,W,D", [(2, 16, 64), (3, 16, 128), (4, 32, 64), (4, 32, 128), (5, 32, 64), (8, 32, 128), (7, 32, 64)])
@pytest.mark.parametrize("S,budget,pool", [(150, 129, 5), (2080, 257, 5), (2113, 64, 7), (4200, 257, 1), (1060, 1000, 131)])
def test_select(monkeypatch, g, W, D, S, budget, pool, page):
    """Scores against the restatement; positions and gathered rows exactly, given the scores."""
    check_select(monkeypatch, 2, 2, g, W, D, S, budget, pool, page, (0, 1))


@pytest.mark.parametrize("B,KH,S", [(50, 8, 700), (133, 3, 530), (64, 4, 2060), (64, 8, 1500), (128, 4, 2100)])
def test_select_of_many_requests(monkeypatch, B, KH, S):
    """Chunks of 512 to 2 304 columns, one and two of them; the last one's rows end inside a column group."""
    check_select(monkeypatch, B, KH, 2, 16, 64, S, 129, 5, 128, (0, B // 2, B - 1))


@pytest.mark.parametrize("B,KH,g,W,D,S", [(52, 4, 8, 32, 64, 700), (19, 8, 8, 32, 128, 521), (12, 8, 4, 32, 128, 1100), (3, 2, 4, 32, 128, 4150)])
def test_select_with_one_workgroup_per_cu(monkeypatch, B, KH, g, W, D, S):
    """Query images that leave room for one workgroup: one chunk of 768 columns, two of 768, many of 256 (over no more columns than the
    bound on differing scores stands for, one in 4 200: over 8 200 it is 5 of 16 336 in whatever chunks)."""
    check_select(monkeypatch, B, KH, g, W, D, S, 129, 5, 128, (0, B - 1))


@pytest.mark.parametrize("g,W,D", [(2, 16, 64), (4, 32, 64), (8, 16, 64), (2, 16, 128), (4, 32, 128), (8, 16, 128)])
@pytest.mark.parametrize("S", [1000, 897 + 64, 1024])
def test_select_in_groups_of_64_columns(monkeypatch, g, W, D, S):
    """256 pairs, an even number of rounds of columns: wavefronts of four column groups, the last of them partly or wholly behind the context."""
    check_select(monkeypatch, 64, 4, g, W, D, S, 129, 5, 128, (0, 63))


# rounds of 16 wavefronts of 32 columns (heads of 64) and of 8 (128): 4 and 8, where a wavefront loads its next 64 columns behind the last
# products, and 7 and 9, the odd numbers from which 64 columns are taken as well; the last columns end inside a group
@pytest.mark.parametrize("g,W,D,S", [(2, 16, 64, 2048), (4, 32, 64, 2040), (8, 16, 64, 4000), (4, 32, 64, 3584), (8, 16, 64, 3500),
                                     (2, 16, 128, 2048), (4, 32, 128, 1792), (8, 16, 128, 2300)])
def test_select_in_groups_of_64_columns_one_after_the_other(monkeypatch, g, W, D, S):
    check_select(monkeypatch, 64, 4, g, W, D, S, 129, 5, 128, (0, 63))


@pytest.mark.parametrize("g,W,D,S", [(2, 16, 64, 1000), (4, 32, 64, 2048), (8, 16, 64, 3584), (2, 16, 128, 1024), (4, 32, 128, 2048), (8, 16, 128, 1792)])
def test_select_in_groups_of_64_columns_of_fp8_pages(g, W, D, S):
    """fp8 pages of the same numbers, with scales that are powers of two: the bits of 16-bit pages that hold them scaled."""
    from magicdec_amd import ops
    B, KH, page, budget = 64, 4, 128, 129
    H, ppr, dpr = KH * g, -(-S // page), budget // page + 1
    gen = torch.Generator().manual_seed(S + g)
    q = torch.randint(-1, 2, (B * W, H, D), generator=gen).bfloat16().to(DEV)
    kv = torch.randint(-1, 2, (B * ppr, 2, KH, page, D), generator=gen).to(DEV)
    scales = tuple(torch.tensor(s, device=DEV) for s in ([0.5, 1.0, 2.0, 0.25], [1.0, 4.0, 0.5, 2.0]))
    table = lambda n: (torch.arange(B * n, dtype=torch.int32, device=DEV), torch.arange(B + 1, dtype=torch.int32, device=DEV) * n)      # noqa: E731
    got = []
    for cache, kw in ((kv.to(torch.float8_e4m3fn), dict(kv_scales=scales)), ((kv * torch.stack(scales).view(1, 2, KH, 1, 1)).bfloat16(), {})):
        draft = torch.zeros(B * dpr, 2, page, KH, D, dtype=torch.bfloat16, device=DEV)
        got.append((*ops.snapkv_select(q, cache, *table(ppr), S, W, budget, 5, draft, *table(dpr), torch.ones(B, dtype=torch.int32, device=DEV),
                                       ops.AttnWorkspace(DEV), return_scores=True, kv_layout="HND", **kw), draft))
    assert all(torch.equal(a, c) for a, c in zip(*got)) and got[0][1].float().isfinite().all() and got[0][2].any()


# accumulators, query image and table of exponentials in one CU's LDS: the most queries a kv head (with the whole table 160 to 170 KB of 160)
@pytest.mark.parametrize("g,W,D", [(32, 8, 128), (30, 8, 128), (28, 8, 128), (16, 16, 128), (32, 8, 64)])
@pytest.mark.parametrize("KH,S", [(1, 1060), (3, 150)])
def test_select_of_many_queries_a_kv_head(monkeypatch, KH, S, g, W, D):
    check_select(monkeypatch, 2, KH, g, W, D, S, 129, 5, 128, (0, 1))


def check_select(monkeypatch, B, KH, g, W, D, S, budget, pool, page, requests):
    from magicdec_amd import ops
    H, ppr, dpr = KH * g, -(-S // page), budget // page + 1
    gen = torch.Generator().manual_seed(S + g)
    q = torch.randint(-1, 2, (B * W, H, D), generator=gen).bfloat16()
    kv = torch.randint(-1, 2, (B * ppr, 2, KH, page, D), generator=gen).bfloat16()
    perm = torch.randperm(B * ppr, generator=gen).int()
    draft = torch.zeros(B * dpr, 2, page, KH, D, dtype=torch.bfloat16, device=DEV)
    args = (torch.arange(B * dpr, dtype=torch.int32, device=DEV), torch.arange(B + 1, dtype=torch.int32, device=DEV) * dpr,
            torch.full((B,), budget - (dpr - 1) * page, dtype=torch.int32, device=DEV))
    idx, sc = ops.snapkv_select(q.to(DEV), kv.to(DEV), perm.to(DEV), torch.arange(B + 1, dtype=torch.int32, device=DEV) * ppr, S, W, budget, pool,
                                draft, *args, ops.AttnWorkspace(DEV), return_scores=True, kv_layout="HND")
    idx, sc, draft = idx.cpu().long(), sc.cpu(), draft.cpu()
    rows = kv[perm.long()].view(B, ppr, 2, KH, page, D).permute(2, 0, 3, 1, 4, 5).reshape(2, B, KH, ppr * page, D)[:, :, :, :S]
    monkeypatch.setattr(mr, "LINEAR_MODE", "fp64")           # correctly rounded scores and weights
    for b in requests:
        want = mr.snapkv_scores(q[b * W:(b + 1) * W], rows[0, b].transpose(0, 1).contiguous(), g, W, pool)
        # fp32 sums of eight rounded weights in another order: at most one of a head's scores or so, by one bf16 step
        off = (sc[b].view(torch.int16).int() - want.view(torch.int16).int()).abs()
        assert int(off.max()) <= 1 and int((off > 0).sum()) <= KH, (b, int((off > 0).sum()))
    for b in requests:
        for h in range(KH):
            v = sc[b, h].float()
            order = torch.sort(v, descending=True, stable=True).indices[:budget - W]          # ties: the lowest positions
            assert torch.equal(idx[b, h], order), (b, h)
            keep = torch.cat([order, torch.arange(S - W, S)])
            got = draft[b * dpr:(b + 1) * dpr, :, :, h].transpose(0, 1).reshape(2, dpr * page, D)[:, :budget]
            assert torch.equal(got, rows[:, b, h][:, keep])


@pytest.mark.parametrize("g,W,D", [(4, 32, 64), (8, 32, 128), (3, 16, 64)])
@pytest.mark.parametrize("power", [-30, -22, -18, -13, 8])
def test_scores_at_the_ends_of_the_table_of_exponentials(g, W, D, power):
    """Scores of one size, 2^power times up to 8 (the tables begin at 2^-23 and 2^-14 and end at 2^9): positions and gathered rows are those of
    the scores that came out, and equal probabilities come out equal -- tiny scores all have the same."""
    from magicdec_amd import ops
    S, budget, KH, page = 1060, 129, 2, 128
    H, ppr = KH * g, -(-S // page)
    gen = torch.Generator().manual_seed(power)
    q = torch.zeros(W, H, D)
    q[:, :, 0] = 2.0 ** power
    keys = torch.randint(1, 9, (ppr * page,), generator=gen).float() * torch.where(torch.rand(ppr * page, generator=gen) < 0.5, -1.0, 1.0)
    kv = torch.randn(ppr, 2, KH, page, D, generator=gen)
    kv[:, 0] = 0
    kv[:, 0, :, :, 0] = keys.view(ppr, 1, page)
    kv, draft = kv.bfloat16(), torch.zeros(2, 2, page, KH, D, dtype=torch.bfloat16, device=DEV)
    one = torch.arange(2, dtype=torch.int32, device=DEV)
    idx, sc = ops.snapkv_select(q.bfloat16().to(DEV), kv.to(DEV), torch.arange(ppr, dtype=torch.int32, device=DEV), one * ppr, S, W, budget, 1, draft, one, one * 2,
                                one[1:], ops.AttnWorkspace(DEV), return_scores=True, kv_layout="HND")
    s = (keys[:S].double() * 2.0 ** power)
    p = torch.softmax(s, 0)[:S - W]                          # (every row has the same scores, but for W x W masked ones of the last few)
    for h in range(KH):
        v = sc[0, h].float().cpu().double()
        # the share of one key: 8 g rows of each chunk, weights and sums rounded to bf16 a few times; masked rows' sums lack up to W keys;
        # weights below 2^-126 are no normal numbers
        assert ((v / (g * W) - p).abs() <= p * (0.04 + 2 * W * p.max()) + 2.0 ** -120).all()
        order = torch.sort(v, descending=True, stable=True).indices[:budget - W]
        assert torch.equal(idx[0, h].cpu().long(), order)
        for k in keys[:S - W].unique():
            assert v[keys[:S - W] == k].unique().numel() == 1
