"""md_linear_f32_few (csrc/f32few.hip) against float64 products, at the edges of its tiles, chunks and slices.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# one step a wavefront, steps that fill no chunk (K = 768: three of four or eight), several chunks; columns that end inside a tile
@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K,wider", [(4, 256, 0), (68, 768, 4), (132, 2048, 0), (12, 8192, 12), (2052, 1280, 0)])
def test_products(M, N, K, wider):
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + N)
    big = torch.full((16 + 4, K + wider), float("nan"), device=DEV)                 # (rows past M stay out of it)
    big[:M] = torch.randn(M, K + wider, device=DEV, generator=g)
    x, w = big[:M, :K], torch.randn(N, K, device=DEV, generator=g)
    ref = x.double() @ w.double().t()
    off = (x.double().abs() @ w.double().abs().t()) * (K * 2.0 ** -24)               # fp32 sums of K terms in any order
    for tile in (0, 8, 16):
        out = ops.linear_f32_few(x, w, tile=tile)
        assert out.shape == (M, N) and ((out.double() - ref).abs() <= off).all()
        assert torch.equal(out[:1], ops.linear_f32_few(x[:1], w, tile=tile))          # a row's bits do not depend on the rows beside it
    x[M // 2, 3] = float("inf")
    out = ops.linear_f32_few(x, w)
    assert out[M // 2].isinf().all() and out.isfinite().all(1).sum() == M - 1


# a shallow K under many columns: fewer tiles than workgroups, some workgroups with a tile more, the last one cut, every depth
@pytest.mark.parametrize("M", [1, 7, 16])
@pytest.mark.parametrize("N,K", [(4100, 256), (4352, 512), (12300, 768), (8200, 1024), (16388, 1280), (20000, 1536), (16384, 1792), (33000, 2048)])
def test_wide(M, N, K):
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + N)
    big = torch.full((16 + 4, K + 4), float("nan"), device=DEV)
    big[:M] = torch.randn(M, K + 4, device=DEV, generator=g)
    x, w = big[:M, :K], torch.randn(N, K, device=DEV, generator=g)
    assert ops.linear_f32_few_supported(M, N, K)
    ref = x.double() @ w.double().t()
    off = (x.double().abs() @ w.double().abs().t()) * (K * 2.0 ** -24)
    out = ops.linear_f32_few(x, w)
    assert out.shape == (M, N) and ((out.double() - ref).abs() <= off).all()
    assert torch.equal(out[:1], ops.linear_f32_few(x[:1], w)) and torch.equal(out, ops.linear_f32_few(x, w))


def test_refused():
    from magicdec_amd import ops
    x, w = torch.randn(4, 256, device=DEV), torch.randn(64, 256, device=DEV)
    assert not any(ops.linear_f32_few_supported(*s) for s in ((4, 8192, 2048), (4, 16384, 2304), (16, 128256, 2048), (17, 64, 256)))
    for call in (lambda: ops.linear_f32_few(torch.randn(17, 256, device=DEV), w), lambda: ops.linear_f32_few(x[:, :128], w[:, :128].contiguous()),
                 lambda: ops.linear_f32_few(x, w[:62].contiguous()), lambda: ops.linear_f32_few(x, w, tile=32), lambda: ops.linear_f32_few(x.double(), w.double()),
                 lambda: ops.linear_f32_few(torch.randn(4, 260, device=DEV)[:, 1:257], w)):
        with pytest.raises((RuntimeError, ValueError, TypeError)):
            call()


def test_shapes_that_the_library_multiplies_faster():
    """They stay there: deep ones of more than 2 048 columns, deep or very narrow ones of nine rows and more over up to 1 024, little more than a
    launch."""
    from magicdec_amd.ops import linear_f32_few_supported as takes
    for M, N, K in ((1, 4096, 4096), (6, 2304, 8192), (9, 1024, 3072), (9, 2048, 3072), (16, 64, 8192), (12, 128, 1536), (1, 1024, 256), (4, 16, 256), (6, 512, 512),
                    (3, 65536, 256)):
        assert not takes(M, N, K), (M, N, K)
    for M, N, K in ((6, 2048, 8192), (6, 2048, 2048), (16, 3072, 2048), (16, 1376, 2048), (16, 2048, 8192), (8, 128, 1536), (4, 128, 256), (16, 3072, 768), (6, 32000, 2048)):
        assert takes(M, N, K), (M, N, K)


@pytest.mark.parametrize("M,N,K", [(4, 2048, 512), (500, 4096, 1024)])
def test_operands_as_they_lie(M, N, K):
    """A weight in columns (as an assigned state dict may bring it) and rows that repeat go to the library, as before these kernels."""
    from magicdec_amd import ops
    from magicdec_amd.Engine.model_layers import LayeredTransformer
    assert ops.linear_f32_few_supported(M, N, K) if M <= 16 else ops.linear_f32_thirds_supported(M, N, K)
    g = torch.Generator(device=DEV).manual_seed(M)
    x, w = torch.randn(M, K, device=DEV, generator=g), torch.randn(N, K, device=DEV, generator=g)
    for a, b in ((x, w.t().contiguous().t()), (x[:1].expand(M, K), w), (x.t().contiguous().t(), w)):
        ref = a.double() @ b.double().t()
        assert ((LayeredTransformer._library(None, a, b).double() - ref).abs() <= (a.double().abs() @ b.double().abs().t()) * (K * 2.0 ** -24)).all()
