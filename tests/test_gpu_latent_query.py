"""md_latent_query (csrc/latent.hip) against md_latent_append and a float64 product of what that leaves.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


# one step a wavefront and several, rows that end inside a tile and inside the append's workgroups, requests without rows and with several, more
# requests than a wavefront has lanes, a layer without a cache of its own, a row past its request's pages
@pytest.mark.parametrize("Q,N,R,RD,new,own", [(256, 32, 64, 32, [1], True), (768, 3072, 512, 64, [1] * 33, True), (512, 96, 40, 24, [3, 0, 17, 1], True),
                                              (1536, 160, 512, 64, [4] * 8, False), (1280, 64, 128, 64, [0] * 70 + [1, 2, 13], True),
                                              (1024, 2048, 96, 32, [1] * 64, True)])
def test_against_append(Q, N, R, RD, new, own):
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(Q + N)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    B, M, page, H, D, VD = len(new), sum(new), 32, 2, 16, 16
    tab = ops.RotaryTable(RD, 10000.0, 500, None, device=DEV)
    spec = ops.LatentSpec(H, D, RD, VD, Q, R, D ** -0.5, 1e-5, tab, rand(H * (D + VD), R).to(BF), (1 + 0.3 * rand(Q)).to(BF), (1 + 0.3 * rand(R)).to(BF) if own else None)
    pos = [(7 * b) % 50 for b in range(B)]
    pos[-1] = 64 - new[-1] + (1 if own and 1 < M < 33 else 0)                              # (the last row may lie past the two pages)
    qo = [0]
    for n in new:
        qo.append(qo[-1] + n)
    order = torch.randperm(2 * B, generator=torch.Generator().manual_seed(2)).tolist()
    where = (ops.StepRows(i32(qo), i32(pos), max(new)), i32(order), i32([2 * b for b in range(B + 1)]), 2)
    z = torch.full((M + 40, Q + R + RD + 8), float("nan"), dtype=BF, device=DEV)
    z[:M] = rand(M, Q + R + RD + 8).to(BF)
    z = z[:M]                                                                           # (rows past M stay out of it)
    w = (rand(N, Q) * Q ** -0.5).to(BF)
    caches = [torch.full((2 * B, page, spec.width), 3.0, dtype=BF, device=DEV) for _ in range(2)]
    pk = ops.PackedWeight(w)
    assert ops.latent_query_supported(z, spec, pk, caches[0])
    ops.page_overflow_count(reset=True)
    cq = ops.latent_append(z, spec, caches[0], *where)
    dropped = ops.page_overflow_count(reset=True)
    q = ops.latent_query(z, spec, pk, caches[1], *where)
    assert dropped == ops.page_overflow_count(reset=True) == (1 if own and 1 < M < 33 else 0)
    assert torch.equal(*caches) and (not own or not caches[0].eq(3.0).all())
    # the scale's sum of squares is of another order: a latent may round the other way (2^-8 of it, rarely), the product sums in fp32
    exact, size = cq.double() @ w.double().t(), cq.double().abs() @ w.double().abs().t()
    near = 2 * Q * 2.0 ** -24 * size + 2.0 ** -8 * exact.abs()
    off = (q.double() - exact).abs()
    assert q.shape == (M, N) and torch.all(off <= near + 2.0 ** -8 * (cq.double().abs().amax(1, keepdim=True) * w.double().abs().amax()) * 4)
    assert (off <= near * 1.01).double().mean() > 0.9


def test_refused():
    from magicdec_amd import ops
    tab = ops.RotaryTable(32, 10000.0, 100, None, device=DEV)
    spec = ops.LatentSpec(2, 16, 32, 16, 256, 64, 0.2, 1e-5, tab, torch.randn(64, 64, device=DEV).to(BF), torch.ones(256, device=DEV).to(BF), torch.ones(64, device=DEV).to(BF))
    cache, pk = torch.zeros(4, 32, spec.width, dtype=BF, device=DEV), ops.PackedWeight(torch.randn(64, 256, device=DEV).to(BF))
    where = (ops.StepRows(i32([0, 65]), i32([0]), 65), i32([0, 1, 2, 3]), i32([0, 4]), 4)
    z = torch.zeros(65, 352, dtype=BF, device=DEV)
    assert not ops.latent_query_supported(z, spec, pk, cache) and ops.latent_query_supported(z[:64], spec, pk, cache)
    assert not ops.latent_query_supported(z[:8].float(), spec, pk, cache) and not ops.latent_query_supported(z[:8, 1:], spec, pk, cache)
    for call in (lambda: ops.latent_query(z, spec, pk, cache, *where), lambda: ops.latent_query(z[:8, :300], spec, pk, cache, *where),
                 lambda: ops.latent_query(z[:8], spec, ops.PackedWeight(torch.randn(64, 512, device=DEV).to(BF)), cache, *where)):
        with pytest.raises((RuntimeError, ValueError, TypeError)):
            call()
