"""A prompt's last portion with its keys split over workgroups (csrc/attn.hip), against the same kernel unsplit.  On the GPU (-m gpu)."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


# rows that fill no wavefront and no workgroup, requests whose keys fill no split (empty ones), more than 64 pages (page numbers are kept 64 at
# a time), groups that begin at any page, both layouts and masks
@pytest.mark.parametrize("H,KH,D,page,lens,past,layout,causal", [
    (32, 8, 128, 128, [33, 33], [2048, 1500], "NHD", True), (32, 8, 64, 64, [70, 1, 45], [5000, 3, 700], "HND", True),
    (16, 4, 128, 128, [129], [9000], "HND", True), (8, 8, 64, 64, [140, 128], [800, 1700], "NHD", False), (28, 4, 128, 64, [19], [4500], "NHD", True)])
def test_against_unsplit(H, KH, D, page, lens, past, layout, causal):
    from magicdec_amd import _lib, ops
    g = torch.Generator(device=DEV).manual_seed(H + D)
    B, tot = len(lens), [n + p for n, p in zip(lens, past)]
    pages, qo, ptr = [-(-t // page) for t in tot], [0], [0]
    for n, k in zip(lens, pages):
        qo.append(qo[-1] + n)
        ptr.append(ptr[-1] + k)
    order = torch.randperm(ptr[-1] + 1, generator=torch.Generator().manual_seed(3)).tolist()[:ptr[-1]]
    shape = (ptr[-1] + 1, 2, page, KH, D) if layout == "NHD" else (ptr[-1] + 1, 2, KH, page, D)
    cache = torch.randn(shape, generator=g, device=DEV).to(BF)
    for b in range(B):                                              # keys and values that were never written
        if tot[b] % page:
            rest = cache[order[ptr[b + 1] - 1]]
            (rest[:, tot[b] % page:] if layout == "NHD" else rest[:, :, tot[b] % page:]).fill_(float("nan"))
    q = (2 * torch.randn(qo[-1], H, D, generator=g, device=DEV)).to(BF)
    ws = ops.AttnWorkspace(DEV)

    def attend(cache, most):
        last = i32([(t - 1) % page + 1 for t in tot])
        return ops.paged_attention(q, cache, i32(qo), i32(order), i32(ptr), last, max(lens), most, ws, causal=causal, kv_layout=layout)

    most, few = max(pages), -(-max(lens) // page)                    # (the bound on the pages decides the plan alone)
    lib = _lib.load()
    assert lib.md_paged_attn_workspace_bytes(B, max(lens), H, KH, D, most, page) > 256 == lib.md_paged_attn_workspace_bytes(B, max(lens), H, KH, D, few, page)
    split, whole = attend(cache, most).double(), attend(cache, few).double()
    size = cache.clone()
    size[:, 1].abs_()
    # weights are rounded to bf16 against other references, sums and the result's rounding follow
    off = 2 * 2.0 ** -9 * attend(size, few).double() * 1.01 + 2.0 ** -8 * whole.abs() + 1e-30
    assert split.isfinite().all() and (split - whole).abs().le(off).all()
    # without room for the parts the keys are not split
    out = torch.empty_like(q)
    kv = _lib.load() and ops._kv_args(cache, None, layout)
    p, last, args = (lambda t: ctypes.c_void_p(t.data_ptr())), i32([(t - 1) % page + 1 for t in tot]), (i32(qo), i32(order), i32(ptr))
    rc = lib.md_paged_attn(p(q), H * D, p(cache), p(out), *map(p, args), p(last), B, max(lens), H, KH, D, page, int(causal), D ** -0.5, most, *kv,
                           None, 0, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0 and torch.equal(out.double(), whole)
