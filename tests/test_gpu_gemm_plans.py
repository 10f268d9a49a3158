"""md_linear where its K slices are uneven (the last one shorter) and with five to seven waves to a workgroup, on row-major and packed,
bf16 and int8 weights: against float64 with the bound of a float32 sum and one rounding.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


@pytest.mark.parametrize("M", [1, 32, 33, 64, 100, 128, 129, 256])
@pytest.mark.parametrize("N,K", [(3584, 4736), (2048, 5632), (2040, 1408), (5120, 2048), (7168, 640), (96, 2176)])
@pytest.mark.parametrize("form", ["rows", "packed", "int8"])
def test_uneven(M, N, K, form):
    from magicdec_amd import ops
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(BF).to(DEV)
    w = torch.randn(N, K, generator=g) * 0.05
    ws, scales = ops.AttnWorkspace(DEV), None
    if form == "int8":
        w8, scales = (w * 400).round().clamp(-127, 127).to(torch.int8).to(DEV), torch.full((N,), 0.0025, dtype=BF, device=DEV)
        exact = (x.double() @ w8.double().t()) * scales.double()
        slack = 2 * K * 2.0 ** -24 * ((x.double().abs() @ w8.double().abs().t()) * scales.double()) + 2.0 ** -8 * exact.abs()
        got = ops.linear(x, ops.PackedWeight(w8), None, scales, False, ws)
    else:
        w = w.to(BF).to(DEV)
        exact = x.double() @ w.double().t()
        slack = 2 * K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
        got = ops.linear(x, ops.PackedWeight(w) if form == "packed" else w, None, None, False, ws)
    assert torch.all((got.double() - exact).abs() <= slack + 2.0 ** -8 * exact.abs() * 1.01)
    if form == "packed" and N % 8 == 0 and ops.linear_add_rmsnorm_supported(M, N, K):
        r, nw = torch.randn(M, N, generator=g).to(BF).to(DEV), torch.ones(N, dtype=BF, device=DEV)
        h, y = ops.linear_add_rmsnorm(x, ops.PackedWeight(w), r, nw, 1e-5, workspace=ws)
        assert all(torch.equal(a, b) for a, b in zip((h, y), ops.add_rmsnorm(r, got, nw, 1e-5)))
        if ops.linear_planes_count("skinny", M, N, K):
            assert torch.all((ops.linear_planes(x, ops.PackedWeight(w), "skinny", ws).planes.double().sum(0) - exact).abs() <= slack)


@pytest.mark.parametrize("M", [1, 33, 128])
@pytest.mark.parametrize("I,K", [(18944, 256), (5632, 512), (9488, 384), (27648, 128)])
def test_gated(M, I, K):
    """Five to seven waves (the bits of four: a wave's columns and slices stay); the last workgroup past the last tile."""
    from magicdec_amd import ops
    g = torch.Generator().manual_seed(M + I)
    x, w = torch.randn(M, K, generator=g).to(BF).to(DEV), (torch.randn(2 * I, K, generator=g) * 0.05).to(BF).to(DEV)
    got = ops.linear(x, ops.PackedWeight(w, swiglu=True), None, None, True, ops.AttnWorkspace(DEV))
    h = x.double() @ w.double().t()
    t = 2 * K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + 2.0 ** -8 * h.abs()
    a, b, ta, tb = h[:, :I], h[:, I:], t[:, :I], t[:, I:]
    exact = torch.nn.functional.silu(a) * b
    tol = (1.1 * ta * (b.abs() + tb) + torch.nn.functional.silu(a).abs() * tb) * 1.01 + 2.0 ** -7 * exact.abs() + 1e-6
    assert torch.all((got.double() - exact).abs() <= tol)
