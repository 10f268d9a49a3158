"""The dispatch rules for linears between the tuned row counts: each rule at the ends of its ranges, through the model's own entry
points, against float64 with the bound of a float32 sum and the roundings to bf16 on the way; and against the route without the rule.
On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
# (rows, N, K, kind, kernel): the first and last rows of each range, the narrowest and widest products, remainders of the tiles
SHAPES = [(33, 20480, 256, "plain", "block"), (128, 32768, 768, "plain", "block"), (65, 32000, 2048, "plain", "block"),
          (1, 14336, 2304, "plain", "fused"), (16, 15008, 2048, "plain", "fused"), (32, 32000, 1024, "plain", "fused"),
          (97, 5120, 4096, "plain", "block"), (256, 8192, 5632, "plain", "block"),
          (3, 14336, 2304, "swiglu", "fused"), (32, 15040, 4096, "swiglu", "fused"),
          (65, 32896, 256, "swiglu", "skinny"), (128, 37888, 512, "swiglu", "skinny"),
          (1, 4096, 8192, "resid", "split"), (32, 4096, 14336, "resid", "split"), (33, 3584, 18944, "resid", "skinny"), (1, 2048, 4224, "resid", "skinny"), (32, 2048, 5632, "resid", "skinny"),
          (33, 2048, 5632, "resid", "fused"), (128, 2048, 4224, "resid", "fused"), (31, 5120, 5120, "resid", "fused"),
          (65, 3584, 3584, "resid", "skinny"), (33, 5120, 5120, "resid", "skinny"), (128, 5120, 4096, "resid", "skinny"), (129, 5120, 5120, "resid", "block"), (255, 5120, 5120, "resid", "block"),
          (1, 2048, 7680, "planes", "skinny"), (64, 1056, 4224, "planes", "skinny"), (65, 2048, 7680, "planes", "skinny"), (256, 2176, 5120, "planes", "skinny"),
          (129, 4096, 4096, "planes", "skinny"), (256, 4096, 4096, "planes", "skinny")]


def model(weight, swiglu):
    from magicdec_amd import ops
    from magicdec_amd.Engine.model_core import Transformer
    m = Transformer.__new__(Transformer)
    torch.nn.Module.__init__(m)
    m._packed, m._released, m.workspace = {id(weight): ops.PackedWeight(weight, swiglu=swiglu)}, set(), ops.AttnWorkspace("cuda")
    return m


@pytest.mark.parametrize("M,N,K,kind,kernel", SHAPES)
def test_rule(M, N, K, kind, kernel):
    from magicdec_amd import ops
    from magicdec_amd.Engine import gemm_policy as g
    if g.mode() != "auto" or g.fused_mode() != "auto" or g.block_mode() != "auto":
        pytest.skip("the environment overrides the rules")
    gen = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=gen).to(BF).cuda()
    w = (torch.randn(N, K, generator=gen) * 0.05).to(BF).cuda()
    resid = torch.randn(M, N, generator=gen).to(BF).cuda()
    lin = torch.nn.Linear(K, N, bias=False, device="meta")
    lin.weight = torch.nn.Parameter(w, requires_grad=False)
    m = model(lin.weight, kind == "swiglu")
    how = g.choose(M, N, K, kind == "swiglu", False, True, kind)
    assert kernel == ("split" if how != "fused" and g.use_split(M, N, K, kind) else how)
    exact = x.double() @ w.double().t()
    # a float32 sum of K products, then one rounding to bf16
    slack = 2 * K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    tol = slack + 2.0 ** -8 * exact.abs()

    def run():
        if kind == "planes":
            planes = ops.linear_planes(x, m._packed[id(lin.weight)], {"split": "tile"}.get(kernel, kernel), m.workspace)
            return planes.planes.double().sum(0)
        if kind == "resid":
            norm = type("Norm", (), {"weight": torch.ones(N, dtype=BF, device="cuda"), "eps": 1e-5})
            return m._proj_add_norm(x, lin, resid, norm, None)[0]
        return m._linear(x, lin if kind == "plain" else None, swiglu_w13=(lin.weight, None) if kind == "swiglu" else None)

    got = run()
    if kind == "planes":
        assert torch.all((got - exact).abs() <= slack)
        return
    if kind == "resid":
        exact = exact + resid.double()
        tol = tol * 1.01 + 2.0 ** -8 * exact.abs()              # ... the residual added in bf16
    if kind == "swiglu":
        a, b = exact[:, :N // 2], exact[:, N // 2:]
        ta, tb = tol[:, :N // 2], tol[:, N // 2:]
        exact = torch.nn.functional.silu(a) * b                 # |d silu| <= 1.1; silu and the product rounded to bf16
        tol = (1.1 * ta * (b.abs() + tb) + torch.nn.functional.silu(a).abs() * tb) * 1.01 + 2.0 ** -7 * exact.abs() + 1e-6
    assert torch.all((got.double() - exact).abs() <= tol * 1.01)
    m._packed = {}                                              # the route without the rule: the row-major weight, in the library
    other = run()
    assert torch.all((got.double() - other.double()).abs() <= 2.02 * tol)
