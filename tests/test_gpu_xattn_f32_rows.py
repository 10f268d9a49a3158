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
