"""md_linear_fused_beside (csrc/tilegemm.hip): two products of the same rows in a launch, against float64.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


# both row tiles of a launch and their ends, one tile beside many and many beside one, a K of one step a wavefront; eight and sixteen wavefronts
@pytest.mark.parametrize("M", [1, 5, 17, 33, 64])
@pytest.mark.parametrize("N,K,N2", [(64, 128, 32), (704, 1024, 1376), (11264, 2048, 96)])
@pytest.mark.parametrize("gelu", [False, True])
def test_against_float64(M, N, K, N2, gelu):
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + N)
    big = torch.full((M + 8, K), float("nan"), dtype=BF, device=DEV)
    big[:M] = torch.randn(M, K, generator=g, device=DEV).to(BF)
    x = big[:M]                                                                          # (rows past M stay out of it)
    w, w2 = ((torch.randn(n, K, generator=g, device=DEV) * K ** -0.5).to(BF) for n in (N, N2))
    assert ops.fused_linear_beside_supported(M, N, K, N2)
    rows = torch.full((M, 8 + N // 2), 7.0, dtype=BF, device=DEV)
    z = ops.fused_linear_beside(x, ops.PackedWeight(w, swiglu=True), rows[:, 8:], ops.PackedWeight(w2), gelu=gelu)
    exact = x.double() @ w2.double().t()
    sums = lambda v: 2 * K * 2.0 ** -24 * (x.double().abs() @ v.double().abs().t())        # fp32 sums of K products
    assert z.shape == (M, N2) and torch.all((z.double() - exact).abs() <= (sums(w2) + 2.0 ** -8 * exact.abs()) * 1.01)
    a, b = (x.double() @ w.double().t()).split(N // 2, 1)
    da, db = sums(w).split(N // 2, 1)
    act = torch.nn.functional.gelu(a, approximate="tanh") if gelu else torch.nn.functional.silu(a)
    # the gate's slope is at most 1.13; SiLU rounds both products and its own result, GELU the last product alone
    r = 0 if gelu else 2.0 ** -8
    off = (1.13 * (da + r * a.abs()) + r * act.abs()) * (b.abs() * (1 + r) + db) + (act.abs() + 1e-6) * (db + r * b.abs())
    assert torch.all((rows[:, 8:].double() - act * b).abs() <= (off + 2.0 ** -8 * (act * b).abs()) * 1.02 + 1e-6)
    assert torch.all(rows[:, :8] == 7.0)


def test_refused():
    from magicdec_amd import ops
    x, w = torch.randn(8, 256, device=DEV).to(BF), torch.randn(64, 256, device=DEV).to(BF)
    gated, plain, out = ops.PackedWeight(w, swiglu=True), ops.PackedWeight(w), torch.empty(8, 32, dtype=BF, device=DEV)
    assert not ops.fused_linear_beside_supported(64, 28672, 4096, 32) and not ops.fused_linear_beside_supported(8, 64, 200, 32)
    for call in (lambda: ops.fused_linear_beside(x, plain, out, plain), lambda: ops.fused_linear_beside(x, gated, out, gated),
                 lambda: ops.fused_linear_beside(x, gated, out[:, :16], plain), lambda: ops.fused_linear_beside(x[:, :128], gated, out, plain)):
        with pytest.raises((RuntimeError, ValueError, TypeError)):
            call()
