"""The tile GEMM's forms for 4 and 16 rows against its 32-row form: a row's bits do not depend on the rows beside it.
On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


@pytest.mark.parametrize("M", [1, 3, 4, 5, 15, 16, 17])
@pytest.mark.parametrize("N,K", [(32, 128), (96, 768), (2048, 2048), (64, 3072), (16384, 1024)])
def test_rows(M, N, K):
    from magicdec_amd import ops
    g = torch.Generator().manual_seed(M + N + K)
    x, r = torch.randn(32, K, generator=g).to(BF).to(DEV), torch.randn(32, N, generator=g).to(BF).to(DEV)
    w = (torch.randn(N, K, generator=g) * 0.05).to(BF).to(DEV)
    p, gated, ws = ops.PackedWeight(w), ops.PackedWeight(w, swiglu=True), ops.AttnWorkspace(DEV)
    big = torch.full((M + 8, K), float("nan"), dtype=BF, device=DEV)
    big[:M] = x[:M]                                              # rows past M stay out of it
    few = big[:M]
    exact = few.double() @ w.double().t()
    slack = (2 * K * 2.0 ** -24 * (few.double().abs() @ w.double().abs().t()) + 2.0 ** -8 * exact.abs()) * 1.01
    got = ops.fused_linear(few, p)
    assert torch.all((got.double() - exact).abs() <= slack)
    assert torch.equal(got, ops.fused_linear(x, p)[:M])
    assert torch.equal(ops.fused_linear(few, gated, swiglu=True), ops.fused_linear(x, gated, swiglu=True)[:M])
    (h, s), (h32, s32) = (ops.fused_linear(a, p, resid=b, want_ssq=True) for a, b in ((few, r[:M]), (x, r)))
    assert torch.equal(h, h32[:M]) and torch.equal(s, s32[:M])
    if K % 256 == 0:                                             # a deferred norm in front
        ssq = x.float().pow(2).view(32, K // 32, 32).sum(-1).contiguous()
        nw = torch.randn(K, generator=g).to(BF).to(DEV)
        a, b = (ops.fused_linear(v, gated, swiglu=True, pro=ops.DeferredNorm(v, q, nw, 1e-5)) for v, q in
                ((few, ssq[:M].contiguous()), (x, ssq)))
        assert torch.equal(a, b[:M])
    if ops.fused_split_supported(M, N, K):
        assert torch.equal(ops.fused_split_linear(few, p, workspace=ws), ops.fused_split_linear(x, p, workspace=ws)[:M])


@pytest.mark.parametrize("D,H,KH", [(64, 4, 2), (128, 5, 1)])
@pytest.mark.parametrize("M,n", [(1, 1), (4, 4), (5, 1), (16, 4)])
def test_rope_append(D, H, KH, M, n):
    from magicdec_amd import ops
    K, N, g = 1024, (H + 2 * KH) * D, torch.Generator().manual_seed(M)
    w = ops.PackedWeight((torch.randn(N, K, generator=g) * 0.05).to(BF).to(DEV))
    x, table = torch.randn(32, K, generator=g).to(BF).to(DEV), ops.RopeTable(512, D, 10000.0, 1.0, device=DEV)
    seen = []
    for rows in (M, 32):
        B = rows // n
        i32 = lambda *a: torch.arange(*a, dtype=torch.int32, device=DEV)
        cache = torch.zeros(B, 2, 128, KH, D, dtype=BF, device=DEV)
        q = ops.fused_qkv_rope_append(x[:rows], w, None, H, KH, D, n, i32(B) + 5, table, cache, i32(B), i32(B + 1),
                                      torch.full((B,), 5 + n, dtype=torch.int32, device=DEV))
        seen.append((q[:M], cache[:M // n]))
    assert all(torch.equal(a, b) for a, b in zip(*seen)) and seen[0][1].abs().sum() > 0
