"""More than 32 query rows a kv head behind a long past, their keys split over workgroups (csrc/attn.hip), against the kernels that take them
without scratch.  On the GPU (-m gpu)."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF, F8 = "cuda:0", torch.bfloat16, torch.float8_e4m3fn


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


# rows that fill no wavefront, group and workgroup, requests whose keys fill no split (empty ones), more than 64 pages (page numbers are kept 64
# at a time), groups that begin at any page, both layouts and masks; few rows on either kernel, many pairs in groups of 32
@pytest.mark.parametrize("H,KH,D,page,lens,past,layout,causal,dtype", [
    (32, 8, 128, 128, [33, 33], [2048, 1500], "NHD", True, BF), (32, 8, 64, 64, [70, 1, 45], [5000, 3, 700], "HND", True, BF),
    (16, 4, 128, 128, [129], [9000], "HND", True, BF), (8, 8, 64, 64, [140, 128], [800, 1700], "NHD", False, BF),
    (28, 4, 128, 64, [19], [4500], "NHD", True, BF), (28, 4, 128, 128, [6, 5, 1], [1200, 9, 3000], "NHD", True, BF),
    (8, 8, 64, 64, [33], [900], "HND", False, BF), (28, 4, 128, 32, [6] * 34, [2100] * 34, "NHD", True, BF),
    (28, 4, 128, 128, [6, 2, 1], [1200, 0, 3000], "NHD", True, F8), (32, 8, 64, 64, [31, 9], [5000, 60], "HND", True, F8)])
def test_against_unsplit(H, KH, D, page, lens, past, layout, causal, dtype):
    from magicdec_amd import _lib, ops
    g = torch.Generator(device=DEV).manual_seed(H + D)
    B, tot, n = len(lens), [n + p for n, p in zip(lens, past)], max(lens)
    pages, qo, ptr = [-(-t // page) for t in tot], [0], [0]
    for k, m in zip(lens, pages):
        qo.append(qo[-1] + k)
        ptr.append(ptr[-1] + m)
    order = torch.randperm(ptr[-1] + 1, generator=torch.Generator().manual_seed(3)).tolist()[:ptr[-1]]
    shape = (ptr[-1] + 1, 2, page, KH, D) if layout == "NHD" else (ptr[-1] + 1, 2, KH, page, D)
    cache = torch.randn(shape, generator=g, device=DEV).to(dtype).to(BF)
    sized = cache.clone()
    sized[:, 1].abs_()
    for b in range(B):                                              # keys and values that were never written
        if tot[b] % page and dtype == BF:
            rest = cache[order[ptr[b + 1] - 1]]
            (rest[:, tot[b] % page:] if layout == "NHD" else rest[:, :, tot[b] % page:]).fill_(float("nan"))
    scales = (0.5 + torch.rand(KH, generator=g, device=DEV), 0.5 + torch.rand(KH, generator=g, device=DEV)) if dtype == F8 else None
    q, most, lib = (2 * torch.randn(qo[-1], H, D, generator=g, device=DEV)).to(BF), max(pages), _lib.load()
    table = [i32(qo), i32(order), i32(ptr), i32([(t - 1) % page + 1 for t in tot])]

    def whole(cache):                                               # no scratch: no split
        out, cache = torch.empty_like(q), cache.to(dtype)
        ptr_ = lambda t: ctypes.c_void_p(t.data_ptr())
        rc = lib.md_paged_attn(ptr_(q), H * D, ptr_(cache), ptr_(out), *map(ptr_, table), B, n, H, KH, D, page, int(causal), D ** -0.5, most,
                               *ops._kv_args(cache, scales, layout), None, 0, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        return out.double()

    assert n * H // KH > 32
    split = ops.paged_attention(q, cache.to(dtype), *table, n, most, ops.AttnWorkspace(DEV), causal=causal, kv_scales=scales, kv_layout=layout).double()
    ref = whole(cache)
    # weights are rounded to bf16 against other references, sums and the result's rounding follow
    off = 2 * 2.0 ** -9 * whole(sized) * 1.01 + 2.0 ** -8 * ref.abs() + 1e-30
    assert split.isfinite().all() and (split - ref).abs().le(off).all()
    assert lib.md_paged_attn_workspace_bytes(B, n, H, KH, D, most, page) > 256 or len(lens) > 30


def test_memory_for_no_scratch(monkeypatch):
    """Rows that need no scratch go without where there is no memory for it; a step's rows, which do, say so.  The workspace stays usable."""
    from magicdec_amd import ops
    B, n, H, KH, D, page, most = 1, 128, 32, 8, 128, 128, 40
    q, cache = torch.randn(n, H, D, device=DEV).to(BF), torch.randn(most, 2, KH, page, D, device=DEV).to(BF)
    table = [i32([0, n]), i32(list(range(most))), i32([0, most]), i32([page])]
    ws, real = ops.AttnWorkspace(DEV), torch.empty
    split = ops.paged_attention(q, cache, *table, n, most, ops.AttnWorkspace(DEV), kv_layout="HND")
    with monkeypatch.context() as m:
        def empty(*size, **kw):
            if kw.get("dtype") == torch.uint8:
                raise torch.OutOfMemoryError("no room")
            return real(*size, **kw)
        m.setattr(torch, "empty", empty)
        whole = ops.paged_attention(q, cache, *table, n, most, ws, kv_layout="HND")
        few = torch.randn(64, H, D, device=DEV).to(BF)
        with pytest.raises(torch.OutOfMemoryError):
            ops.paged_attention(few, cache, i32(list(range(0, 65, 8))), i32([0] * 8 * most), i32([most * b for b in range(9)]), i32([page] * 8), 8, most, ws,
                                kv_layout="HND")
    assert ws._retired == [] and ws.buf.numel() == 1 << 20
    assert (whole.float() - split.float()).norm() <= 0.01 * whole.float().norm()
    assert torch.equal(ops.paged_attention(q, cache, *table, n, most, ws, kv_layout="HND"), split)
