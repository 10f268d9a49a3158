"""md_linear_f32 (csrc/f32gemm.hip) against float64 products, at the edges of its tiles.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# one row, tiles' edges in rows and columns, one step of 32 and an odd number of them, rows wider than K, several tiles a CU
@pytest.mark.parametrize("M,N,K,wider", [(1, 4, 32, 0), (33, 68, 96, 4), (64, 128, 64, 0), (65, 132, 32, 12), (127, 1000, 160, 0), (257, 60, 2048, 0),
                                         (1500, 3076, 96, 0)])
def test_products(M, N, K, wider):
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, K + wider, device=DEV, generator=g)[:, :K]
    w = torch.randn(N, K, device=DEV, generator=g)
    ref = x.double() @ w.double().t()
    off = (x.double().abs() @ w.double().abs().t()) * (K * 2.0 ** -24)               # fp32 sums of K terms in any order
    first = None
    for tile in (0, 64128, 64064, 32064):
        out = ops.linear_f32(x, w, tile=tile)
        assert out.shape == (M, N) and ((out.double() - ref).abs() <= off).all()
        first = out if first is None else first
        assert torch.equal(out, first)                                                # one order of the sums, whatever the tile
    x[M // 2, 3] = float("nan")
    out = ops.linear_f32(x, w)
    assert out[M // 2].isnan().all() and out.isnan().any(1).sum() == 1


def test_refused():
    from magicdec_amd import ops
    x, w = torch.randn(100, 64, device=DEV), torch.randn(64, 64, device=DEV)
    for call in (lambda: ops.linear_f32(x[:, :48], w[:, :48].contiguous()), lambda: ops.linear_f32(x, w[:62].contiguous()),
                 lambda: ops.linear_f32(x, w, tile=16016), lambda: ops.linear_f32(x.double(), w.double()),
                 lambda: ops.linear_f32(torch.randn(100, 66, device=DEV)[:, 1:65], w)):
        with pytest.raises((RuntimeError, ValueError, TypeError)):
            call()
