"""Decode attention at request counts around the rule that splits keys over workgroups (and, in fp8, picks the wavefronts), against
float64.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("B,KH,ctx,n", [(1, 1, 4161, 1), (5, 4, 4161, 4), (7, 8, 1500, 2), (28, 8, 3300, 1), (32, 8, 700, 4), (33, 8, 4161, 1),
                                        (40, 8, 4161, 2), (41, 8, 4161, 1), (33, 8, 8300, 1)])
def test_splits(B, KH, ctx, n, fp8):
    check(B, KH, ctx, n, fp8)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("B,KH,ctx,n", [(21, 4, 2100, 4), (44, 8, 8300, 1), (48, 8, 8300, 2), (49, 8, 8300, 1)])
def test_splits_of_an_xcd(B, KH, ctx, n, fp8):
    """A pair's workgroups lie on one XCD: 11 pairs on some of them take two splits, 44 and 48 two, 49 none."""
    check(B, KH, ctx, n, fp8)


def check(B, KH, ctx, n, fp8):
    """bf16 weights of the values: |error| <= 2^-8 of the weighted |v|, plus the output's own rounding; fp32 sums elsewhere."""
    from magicdec_amd import ops
    D, g, pp = 64, 4, -(-ctx // 128)
    gen = torch.Generator(device=DEV).manual_seed(B + ctx)
    cache = torch.randn(B * pp, 2, KH, 128, D, device=DEV, generator=gen).to(torch.float8_e4m3fn if fp8 else torch.bfloat16)
    q = torch.randn(B * n, KH * g, D, device=DEV, generator=gen).bfloat16()
    scales = (torch.full((KH,), 0.7, device=DEV), torch.full((KH,), 1.3, device=DEV)) if fp8 else None
    last = torch.full((B,), ctx - (pp - 1) * 128, dtype=torch.int32, device=DEV)
    got = ops.paged_attention(q, cache, torch.arange(B + 1, dtype=torch.int32, device=DEV) * n, torch.arange(B * pp, dtype=torch.int32, device=DEV),
                              torch.arange(B + 1, dtype=torch.int32, device=DEV) * pp, last, n, pp, ops.AttnWorkspace(DEV), kv_scales=scales,
                              kv_layout="HND").double()
    for b in {0, B // 2, B - 1}:
        rows = cache[b * pp:(b + 1) * pp].double().permute(1, 2, 0, 3, 4).reshape(2, KH, pp * 128, D)[:, :, :ctx]
        k, v = rows[0] * (0.7 if fp8 else 1.0), rows[1] * (1.3 if fp8 else 1.0)
        for h in range(KH):
            x = q[b * n:(b + 1) * n, h * g:(h + 1) * g].double().reshape(n * g, D)
            s = (x @ k[h].t()) * D ** -0.5
            s = s.view(n, g, ctx).masked_fill(torch.arange(ctx, device=DEV) > torch.arange(ctx - n, ctx, device=DEV).view(n, 1, 1), float("-inf"))
            p = torch.softmax(s, -1)
            want, size = p @ v[h], p @ v[h].abs()
            out = got[b * n:(b + 1) * n, h * g:(h + 1) * g]
            assert bool(((out - want).abs() <= 2.0 ** -8 * (size + want.abs()) + 1e-6).all()), (b, h)
