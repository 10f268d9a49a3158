"""The 32-bit prompt attention that gives a wavefront its own rows (csrc/xattn_f32.hip), against float64.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def reference(qkv, spec, n, pos, past):
    """float64: (output, bound of the error of 32-bit arithmetic) of one sequence; past: its earlier (k, v) rows"""
    H, KH, D, DV = spec.H, spec.KH, spec.D, spec.DV
    q, k, v = qkv.double().split([H * D, KH * D, KH * DV], 1)
    k, v = torch.cat([past[0], k]).view(-1, KH, D).repeat_interleave(H // KH, 1), torch.cat([past[1], v]).view(-1, KH, DV).repeat_interleave(H // KH, 1)
    q = q.view(n, H, D)
    at, key = torch.arange(pos, pos + n, device=DEV)[:, None], torch.arange(pos + n, device=DEV)[None]
    seen = (key <= at) & (key >= at // spec.chunk * spec.chunk if spec.chunk else key >= 0)
    s, off = torch.einsum("nhd,khd->hnk", q, k) * spec.scale, torch.einsum("nhd,khd->hnk", q.abs(), k.abs()) * spec.scale * (D + 4) * 2.0 ** -24
    if spec.r1 is not None:
        far = torch.log1p(spec.r2.double()[:, None, None] * (at - key).clamp(min=0))
        s, off = s - spec.r1.double()[:, None, None] * far, off + spec.r1.double()[:, None, None] * (far + 1) * 2.0 ** -21
    off = (off + s.abs() * 2.0 ** -22).masked_fill(~seen, 0).amax(2)                       # of a score, its log2 and the reference taken off
    s = s.masked_fill(~seen, -torch.inf)
    if spec.sink:
        w = torch.softmax(torch.cat([s, torch.zeros(H, n, 1, device=DEV, dtype=s.dtype)], 2), 2)[..., :-1]
    else:
        w = torch.softmax(s, 2)
    none = torch.zeros((), device=DEV, dtype=torch.float64)
    out = torch.stack([(w[h][:, :, None] * torch.where(seen[:, :, None], v[None, :, h], none)).sum(1) for h in range(H)], 1)
    size = torch.stack([w[h] @ v[:, h].nan_to_num(0, 0, 0).abs() for h in range(H)], 1)
    return out.reshape(n, -1), (size * (2 * off.t()[:, :, None] + (pos + n + 16) * 2.0 ** -23) + 1e-37).reshape(n, -1)


# rows that end inside a wavefront and a workgroup, heads that no row tile is a multiple of, odd sizes, chunks, long pasts (key splits),
# scores that grow by far more than the reference may lag, and scores of a row that are all very low
@pytest.mark.parametrize("H,KH,D,DV,lens,pos,chunk,kind", [
    (32, 8, 64, 64, [17, 70, 301], [0, 0, 0], 0, "bias"), (12, 4, 48, 64, [150, 3, 161], [5, 0, 40], 0, "sink"), (10, 2, 128, 128, [129, 200], [0, 31], 64, "bias"),
    (16, 16, 64, 64, [65, 127], [0, 900], 0, "grow"), (16, 4, 128, 96, [210, 33], [0, 700], 0, "low"), (8, 8, 32, 32, [400], [1], 100, "none")])
def test_against_float64(H, KH, D, DV, lens, pos, chunk, kind):
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(H + D)
    bias = [torch.rand(H, device=DEV, generator=g) * 4 for _ in range(2)] if kind == "bias" else [None, None]
    spec = ops.XattnSpec(H, KH, D, DV, D ** -0.5, 1e-6, chunk=chunk, sink=kind == "sink", r1=bias[0], r2=bias[1])
    page, total = 32, [n + p for n, p in zip(lens, pos)]
    pages, ptr = [-(-t // page) for t in total], [0]
    for n in pages:
        ptr.append(ptr[-1] + n)
    order = torch.randperm(ptr[-1] + 2, generator=torch.Generator().manual_seed(1)).tolist()
    kc, vc = (torch.full((len(order), KH, page, ops.head_pad(w)), float("nan"), device=DEV) for w in (D, DV))
    ws, outs = ops.AttnWorkspace(DEV), []

    def attend(rows, n, at):
        qo = [0]
        for x in n:
            qo.append(qo[-1] + x)
        return ops.extended_attention(torch.cat(rows), spec, kc, vc, ops.StepRows(i32(qo), i32(at), max(n)), i32(order[:ptr[-1]]), i32(ptr), max(pages), ws)

    qkv = []
    for t in total:
        x = torch.randn(t, H * D + KH * (D + DV), device=DEV, generator=g)
        if kind == "grow":                                                      # later keys win, by hundreds
            x[:, H * D:(H + KH) * D] = torch.linspace(-1, 40, t, device=DEV)[:, None] * x[:1, :D].repeat(1, KH)
            x[:, :H * D] = x[:1, :D].repeat(t, H) * 4
        elif kind == "low":
            x[:, :H * D], x[:, H * D:(H + KH) * D] = x[:, :H * D].abs() * 8, -x[:, H * D:(H + KH) * D].abs() * 8
        qkv.append(x)
    for b, p in enumerate(pos):                                                 # the past, a sequence at a time
        if p:
            attend([q[:p] if i == b else q[:0] for i, q in enumerate(qkv)], [p if i == b else 0 for i in range(len(lens))], [0] * len(lens))
    qkv[0][-1, -DV:] = float("inf")                                             # a value that only the last row sees
    out = attend([q[p:] for q, p in zip(qkv, pos)], lens, pos).split(lens)
    for q, n, p, o in zip(qkv, lens, pos, out):
        past = q[:p, H * D:].double().split([KH * D, KH * DV], 1)
        ref, off = reference(q[p:], spec, n, p, past)
        last = ref.isinf()
        assert torch.equal(o.isinf(), last) and (o[~last].double() - ref[~last]).abs().le(off[~last]).all(), (o.double() - ref)[~last].abs().max()


# steps of a row or a few: pasts around the first that is split, whose splits are two tiles, more than eight splits to merge, splits of
# several tiles, wide heads, a chunk that begins inside a tile; sequences of unequal lengths, whose last splits have no key
@pytest.mark.parametrize("H,KH,D,DV,lens,pos,chunk,kind", [
    (32, 8, 64, 64, [1, 1, 1], [0, 255, 254], 0, "bias"), (32, 8, 64, 64, [1, 1], [319, 3], 0, "none"), (8, 2, 64, 64, [4, 1, 1], [1500, 600, 40], 0, "sink"),
    (16, 4, 64, 48, [1], [2300], 1000, "bias"), (8, 4, 128, 128, [2, 1, 1], [127, 160, 900], 0, "bias"), (4, 1, 256, 256, [1, 1], [129, 700], 0, "sink"),
    (16, 16, 256, 192, [1, 1, 1], [800, 60, 300], 0, "none")])
def test_steps_against_float64(H, KH, D, DV, lens, pos, chunk, kind):
    test_against_float64(H, KH, D, DV, lens, pos, chunk, kind)


def attend_alone(q, k, v, spec, page=32):
    """One sequence from its first token: q [n, H, D], k [n, KH, D], v [n, KH, DV]"""
    from magicdec_amd import ops
    n, pages = q.shape[0], -(-q.shape[0] // page)
    caches = [torch.zeros(pages, spec.KH, page, ops.head_pad(w), device=DEV) for w in (spec.D, spec.DV)]
    return ops.extended_attention(torch.cat([x.flatten(1) for x in (q, k, v)], 1), spec, *caches, ops.StepRows(i32([0, n]), i32([0]), n), i32(list(range(pages))),
                                  i32([0, pages]), pages, ops.AttnWorkspace(DEV)).view(n, spec.H, spec.DV)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("score", [3.0, 1e6, -1e9, -1e28])
def test_equal_scores_weigh_the_same_whatever_their_size(D, score):
    """Tiles of equal scores: each value of the past counts once.  (A scaled score that is part of a fused operation in one tile and rounded
    in another is half a step of its own size off.)"""
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(D)
    H, KH, n = 32, 16, 300
    spec = ops.XattnSpec(H, KH, D, D, D ** -0.5, 1e-6)
    q, k = torch.ones(n, H, D, device=DEV), torch.full((n, KH, D), score / D * D ** 0.5, device=DEV)
    v = torch.randn(n, KH, D, device=DEV, generator=g)
    out, count = attend_alone(q, k, v, spec).double(), torch.arange(1, n + 1, device=DEV)[:, None, None]
    mean, size = ((x.double().cumsum(0) / count).repeat_interleave(H // KH, 1) for x in (v, v.abs()))
    assert (out - mean).abs().le(size * (n + 16) * 2.0 ** -23).all()


@pytest.mark.parametrize("above", [0.0, 1.9, 3.9, 30.0])
def test_values_near_the_end_of_the_range(above):
    """Values whose sum over the keys is a number as long as weights are at most 1, behind a tile whose scores are lower by `above` (log2)."""
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(int(above))
    H, KH, n, D = 32, 16, 400, 64
    spec = ops.XattnSpec(H, KH, D, D, D ** -0.5, 1e-6)
    q, k = torch.ones(n, H, D, device=DEV), torch.zeros(n, KH, D, device=DEV)
    k[32:] = above / 1.4426950408889634 / D * D ** 0.5
    v = (torch.rand(n, KH, D, device=DEV, generator=g) - 0.25) * 1.5e36
    out = attend_alone(q, k, v, spec).double()
    s = (torch.einsum("nhd,khd->hnk", q[:, ::2].double(), k.double()) * spec.scale).masked_fill(torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1), -torch.inf)
    w = torch.softmax(s, 2)
    ref, size = (torch.einsum("hnk,khd->nhd", w, x.double()).repeat_interleave(2, 1) for x in (v, v.abs()))
    assert out.isfinite().all() and (out - ref).abs().le(size * (n + 64) * 2.0 ** -22).all()


@pytest.mark.parametrize("D", [64, 128])
def test_error_of_a_biased_prompt(D):
    """Against float64 no further off, as a 2-norm, than the kernel of row groups of 16, which takes each head alone (the order in which the
    bias and the reference come off a score is worth a fifth of the error)."""
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(D)
    H, n = 16, 700
    b = [torch.rand(H, device=DEV, generator=g) * 2 for _ in range(2)]
    spec = ops.XattnSpec(H, H, D, D, D ** -0.5, 1e-6, r1=b[0], r2=b[1])
    qkv = torch.randn(n, 3 * H * D, device=DEV, generator=g)
    heads = [x.view(n, H, D) for x in qkv.chunk(3, 1)]
    none = torch.zeros(0, H * D, device=DEV, dtype=torch.float64)
    ref = reference(qkv, spec, n, 0, (none, none))[0].view(n, H, D)
    alone = [attend_alone(*(x[:, h:h + 1].contiguous() for x in heads), ops.XattnSpec(1, 1, D, D, D ** -0.5, 1e-6, r1=b[0][h:h + 1], r2=b[1][h:h + 1])) for h in range(H)]
    assert (attend_alone(*heads, spec).double() - ref).norm() <= 1.03 * (torch.cat(alone, 1).double() - ref).norm()
