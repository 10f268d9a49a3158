"""md_linear_few (csrc/tilegemm.hip): a row to sixteen on tiles of 16 columns, against float64 products and the 32-column form.
On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


def bound(x, w, exact):
    """fp32 sums of K products, one rounding to bf16."""
    K = x.shape[1]
    return (2 * K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + 2.0 ** -8 * exact.abs()) * 1.01


# one tile pair; steps that fill no chunk (K = 768, 1 280), a ring (2 048) and several (14 336); a round of the chip
@pytest.mark.parametrize("M", [1, 4, 5, 16])
@pytest.mark.parametrize("N,K", [(32, 256), (96, 768), (64, 1280), (4096, 2048), (160, 14336)])
def test_products_and_epilogues(M, N, K):
    from magicdec_amd import ops
    g = torch.Generator().manual_seed(M + N + K)
    big = torch.full((M + 8, K), float("nan"), dtype=BF, device=DEV)
    big[:M] = torch.randn(M, K, generator=g).to(BF).to(DEV)
    x, r = big[:M], torch.randn(M, N, generator=g).to(BF).to(DEV)                        # (rows past M stay out of it)
    w, bias = (torch.randn(N, K, generator=g) * 0.05).to(BF).to(DEV), torch.randn(N, generator=g).to(BF).to(DEV)
    p, gated = ops.PackedWeight(w), ops.PackedWeight(w, swiglu=True)
    exact = x.double() @ w.double().t()
    plain = ops.fused_linear(x, p, few=True)
    assert torch.all((plain.double() - exact).abs() <= bound(x, w, exact))
    with_bias = exact + bias.double()
    assert torch.all((ops.fused_linear(x, p, bias, few=True).double() - with_bias).abs() <= bound(x, w, with_bias) + 2.0 ** -8 * bias.double().abs())
    # the residual add and its sums are those of what the plain product returns
    h, ssq = ops.fused_linear(x, p, resid=r, want_ssq=True, few=True)
    assert torch.equal(h, plain + r) and ssq.shape == (M, N // 16)
    assert torch.allclose(ssq, h.float().square().view(M, N // 16, 16).sum(-1), rtol=2e-6, atol=0)
    # the gated epilogue from the halves' own products
    act = ops.fused_linear(x, gated, swiglu=True, few=True)
    a, b = plain[:, :N // 2].float(), plain[:, N // 2:].float()
    want = torch.nn.functional.silu(a.double()) * b.double()
    assert torch.all((act.double() - want).abs() <= 2.0 ** -7 * want.abs() + 1e-30)
    # the activation takes the sum before its rounding (2^-9 of z, and xielu's slope is at most 1 + 2 * 0.9 |z| there), then rounds once
    xi, z = torch.tensor([0.3, -0.2], device=DEV), plain.float()
    off = (ops.fused_linear(x, p, xielu=xi, few=True).float() - ops.xielu(plain, xi).float()).abs()
    assert torch.all(off <= 2.0 ** -8 * z.abs() * (1 + 1.8 * z.abs()) + 2.0 ** -7 * ops.xielu(plain, xi).float().abs() + 1e-30)


@pytest.mark.parametrize("M", [1, 4, 5, 16])
@pytest.mark.parametrize("N,K", [(96, 768), (64, 8192), (8192, 1024)])
def test_deferred_norm(M, N, K):
    """A norm in front from either kind of partial sums (more than four a lane at K = 8 192), also of the wide plain product on 32 columns
    and of the kernels that take 32-column sums; the norm's own launch differs in the order of its sum of squares."""
    from magicdec_amd import ops
    g = torch.Generator().manual_seed(M + N)
    x = torch.randn(M, K, generator=g).to(BF).to(DEV)
    w, nw = (torch.randn(N, K, generator=g) * 0.05).to(BF).to(DEV), torch.randn(K, generator=g).to(BF).to(DEV)
    p, gated, ws = ops.PackedWeight(w), ops.PackedWeight(w, swiglu=True), ops.AttnWorkspace(DEV)
    y = ops.rmsnorm(x, nw, 1e-5)
    close = lambda got, want: bool(((got.float() - want.float()).abs() <= 2.0 ** -6 * want.float().abs() + 2.0 ** -6 * want.float().std()).all())
    for cols in (16, 32):
        pro = ops.DeferredNorm(x, x.float().square().view(M, K // cols, cols).sum(-1).contiguous(), nw, 1e-5)
        assert close(ops.fused_linear(x, p, few=True, pro=pro), ops.fused_linear(y, p, few=True))
        assert close(ops.fused_linear(x, gated, swiglu=True, few=True, pro=pro), ops.fused_linear(y, gated, swiglu=True, few=True))
        assert close(ops.fused_linear(x, gated, swiglu=True, pro=pro), ops.fused_linear(y, gated, swiglu=True))
        assert close(ops.linear(x, gated, swiglu=True, workspace=ws, pro=pro), ops.linear(y, gated, swiglu=True, workspace=ws))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D,H,KH", [(64, 4, 2), (128, 5, 1)])
@pytest.mark.parametrize("M,n", [(1, 1), (4, 4), (5, 1), (16, 4)])
def test_rope_append(D, H, KH, M, n, fp8):
    from magicdec_amd import ops
    K, N, g, B = 1024, (H + 2 * KH) * D, torch.Generator().manual_seed(M), M // n
    wt = (torch.randn(N, K, generator=g) * 0.05).to(BF).to(DEV)
    w, x = ops.PackedWeight(wt), torch.randn(M, K, generator=g).to(BF).to(DEV)
    table, i32 = ops.RopeTable(512, D, 10000.0, 1.0, device=DEV), lambda *a: torch.arange(*a, dtype=torch.int32, device=DEV)
    scales = (torch.full((KH,), 0.02, device=DEV),) * 2 if fp8 else None
    kind = torch.float8_e4m3fn if fp8 else BF
    pages = (i32(B), i32(B + 1), torch.full((B,), 5 + n, dtype=torch.int32, device=DEV))
    caches = [torch.zeros(B, 2, KH, 128, D, dtype=BF, device=DEV).to(kind) for _ in range(2)]
    q = ops.fused_qkv_rope_append(x, w, None, H, KH, D, n, i32(B) + 5, table, caches[0], *pages, kv_scales=scales, kv_layout="HND", few=True)
    z = ops.fused_linear(x, w, few=True)
    want = ops.rope_append(z[:, :H * D].unflatten(1, (H, D)), z[:, H * D:(H + KH) * D].unflatten(1, (KH, D)), z[:, (H + KH) * D:].unflatten(1, (KH, D)),
                           i32(B + 1) * n, i32(B) + 5, table, caches[1], *pages, n_max=n, kv_scales=scales, kv_layout="HND")
    assert torch.equal(q, want) and torch.equal(*(c.view(torch.uint8) for c in caches)) and caches[0].float().abs().sum() > 0


def test_refused():
    from magicdec_amd import ops
    p = ops.PackedWeight(torch.randn(64, 256, device=DEV).to(BF))
    odd = ops.PackedWeight(torch.randn(64, 384, device=DEV).to(BF))
    for call in (lambda: ops.fused_linear(torch.randn(17, 256, device=DEV).to(BF), p, few=True),
                 lambda: ops.fused_linear(torch.randn(4, 384, device=DEV).to(BF), odd, few=True)):
        with pytest.raises(RuntimeError):
            call()


def test_rule():
    from magicdec_amd.Engine.gemm_policy import use_few
    assert use_few(1, 768, 3072) and use_few(16, 4096, 4096) and use_few(4, 4096, 14336)
    for M, N, K in ((17, 768, 3072), (1, 4128, 4096), (1, 768, 768), (1, 992, 8192), (1, 2048, 1152), (0, 768, 3072)):
        assert not use_few(M, N, K)


def test_rule_ends_where_either_form_is_a_handful_of_workgroups():
    from magicdec_amd.Engine.gemm_policy import use_few
    assert use_few(1, 160, 1536) and not any(use_few(M, N, 1536) for M in (1, 16) for N in (32, 128))
