"""md_linear_f32_thirds (csrc/f32thirds.hip) against float64 products, at the edges of its tiles.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TILES = (0, 256256, 192256, 160256, 128256, 256128, 192128, 128128, 64128)


# one row, tiles' edges in rows and columns, one to three steps of 32, rows wider than K, several tiles a CU
@pytest.mark.parametrize("M,N,K,wider", [(1, 4, 32, 0), (33, 68, 96, 4), (64, 128, 64, 0), (65, 132, 32, 12), (127, 1000, 160, 0), (257, 60, 2048, 0),
                                         (161, 260, 128, 0), (1500, 3076, 96, 0)])
def test_products(M, N, K, wider):
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, K + wider, device=DEV, generator=g)[:, :K] * 2.0 ** torch.randint(-12, 13, (M, 1), device=DEV, generator=g)
    w = torch.randn(N, K, device=DEV, generator=g)
    ref = x.double() @ w.double().t()
    off = (x.double().abs() @ w.double().abs().t()) * (K * 2.0 ** -24)               # fp32 sums of K terms in any order
    first = None
    for tile in TILES:
        out = ops.linear_f32_thirds(x, w, tile=tile)
        assert out.shape == (M, N) and ((out.double() - ref).abs() <= off).all()
        first = out if first is None else first
        assert torch.equal(out, first)                                                # one order of the sums, whatever the tile
    x[M // 2, 3] = float("nan")
    out = ops.linear_f32_thirds(x, w)
    assert out[M // 2].isnan().all() and out.isnan().any(1).sum() == 1


def test_no_further_off_than_the_fp32_instruction():
    """The error against 64 bits of a deep product, as a norm: what the parts leave out must not show beside what 32-bit sums round."""
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(0)
    x, w = torch.randn(600, 4096, device=DEV, generator=g), torch.randn(512, 4096, device=DEV, generator=g)
    ref = x.double() @ w.double().t()
    assert (ops.linear_f32_thirds(x, w).double() - ref).norm() <= (ops.linear_f32(x, w).double() - ref).norm()


@pytest.mark.parametrize("K", [256, 2048])
@pytest.mark.parametrize("kind", ["normal", "positive", "shifted", "outliers", "zeros"])
def test_error_beside_the_fp32_instruction_s(kind, K):
    """The same over other distributions.  Zeros cost the fp32 instruction's sums no rounding, six parts of the others do."""
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(K)
    x, w = torch.randn(512, K, device=DEV, generator=g), torch.randn(512, K, device=DEV, generator=g)
    if kind == "positive":
        x, w = torch.rand(512, K, device=DEV, generator=g), torch.rand(512, K, device=DEV, generator=g)
    elif kind == "shifted":
        x, w = x + 0.25, w + 0.25
    elif kind == "outliers":
        x[:, ::97] *= 100
    elif kind == "zeros":
        x = x.relu()
    ref = x.double() @ w.double().t()
    assert (ops.linear_f32_thirds(x, w).double() - ref).norm() <= (1.3 if kind == "zeros" else 1) * (ops.linear_f32(x, w).double() - ref).norm()


@pytest.mark.parametrize("K", [32, 2048])
@pytest.mark.parametrize("sign", [1, -1])
def test_operands_whose_rests_are_as_large_as_they_can_be(K, sign):
    """What the six products leave out is then 2^-24 of each term, and of one sign."""
    from magicdec_amd import ops
    v = 1 + 2.0 ** -8 - 2.0 ** -17 + 2.0 ** -23
    x, w = torch.full((70, K), v, device=DEV), torch.full((132, K), sign * v, device=DEV)
    ref = x.double() @ w.double().t()
    assert ((ops.linear_f32_thirds(x, w).double() - ref).abs() <= ref.abs() * ((K + 1) * 2.0 ** -24)).all()


@pytest.mark.parametrize("power", [-100, -110, -116, -122, -130, 100])
@pytest.mark.parametrize("small", ["x", "w"])
def test_numbers_of_any_size(power, small):
    """Parts are multiples of 2^-133: each number is held to 2^-134, beside what 32-bit sums round (of results below 2^-126 to 2^-150)."""
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(-power)
    K = 256
    x, w = torch.randn(130, K, device=DEV, generator=g), torch.randn(132, K, device=DEV, generator=g)
    if small == "x":
        x = (x.double() * 2.0 ** power).float()
    else:
        w = (w.double() * 2.0 ** power).float()
    a, b = x.double().abs(), w.double().abs()
    held = 2.0 ** -134 * (a.sum(1)[:, None] + b.sum(1)[None]) * 1.01
    off = (a @ b.t()) * (K * 2.0 ** -24) + held + K * 2.0 ** -149
    assert ((ops.linear_f32_thirds(x, w).double() - x.double() @ w.double().t()).abs() <= off).all()


def test_infinities_and_numbers_that_round_to_them():
    from magicdec_amd import ops
    x, w = torch.ones(70, 64, device=DEV), torch.ones(132, 64, device=DEV)
    w[:, 1] = 0.75
    x[3, 5], x[4, 6], x[5, :2] = float("inf"), float("-inf"), torch.tensor([float("inf"), float("-inf")])
    x[6, 7], w[:, 7], w[9, 8], w[10, 9] = 3.4e38, 0.5, float("inf"), 3.4e38
    out, ref = ops.linear_f32_thirds(x, w), (x.double() @ w.double().t())
    assert torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.isinf(), ref.isinf() | (ref.abs() > 3.4028236e38))
    fine = out.isfinite()
    assert ((out.double() - ref).abs()[fine] <= ref.abs()[fine] * 64 * 2.0 ** -24).all() and torch.equal(out[out.isinf()] > 0, ref[out.isinf()] > 0)


def test_rows_in_several_calls(monkeypatch):
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(1)
    x, w = torch.randn(700, 64, device=DEV, generator=g), torch.randn(68, 64, device=DEV, generator=g)
    whole = ops.linear_f32_thirds(x, w)
    monkeypatch.setattr(ops, "THIRDS_BYTES", 300 * 64 * 6)
    assert torch.equal(ops.linear_f32_thirds(x, w), whole)


def test_more_rows_than_a_call_takes():
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(2)
    x, w = torch.randn(16 * 65535 + 100, 32, device=DEV, generator=g), torch.randn(4, 32, device=DEV, generator=g)
    out = ops.linear_f32_thirds(x, w)
    for at in (0, 4095 * 256 - 64, x.shape[0] - 128):
        assert torch.equal(out[at:at + 128], ops.linear_f32_thirds(x[at:at + 128], w))


def room(monkeypatch, nbytes):
    """torch.empty finds no memory once `nbytes` are asked for in all."""
    real, left = torch.empty, [nbytes]

    def empty(*size, **kw):
        t = real(*size, **dict(kw, device="meta"))
        if t.numel() * t.element_size() > left[0]:
            raise torch.OutOfMemoryError("no room")
        left[0] -= t.numel() * t.element_size()
        return real(*size, **kw)
    monkeypatch.setattr(torch, "empty", empty)


@pytest.mark.parametrize("M,N,K", [(256, 512, 64), (256, 64, 512)])
def test_memory_for_the_result_alone(monkeypatch, M, N, K):
    """Scratch larger than the result or smaller: with room for either, not both, the rows are multiplied without it."""
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(N)
    x, w = torch.randn(M, K, device=DEV, generator=g), torch.randn(N, K, device=DEV, generator=g)
    want = ops.linear_f32(x, w)
    room(monkeypatch, max(4 * M * N, 6 * M * K))
    assert torch.equal(ops.linear_f32_thirds(x, w), want)


def test_refused():
    from magicdec_amd import ops
    x, w = torch.randn(100, 64, device=DEV), torch.randn(64, 64, device=DEV)
    for call in (lambda: ops.linear_f32_thirds(x[:, :48], w[:, :48].contiguous()), lambda: ops.linear_f32_thirds(x, w[:62].contiguous()),
                 lambda: ops.linear_f32_thirds(x, w, tile=16016), lambda: ops.linear_f32_thirds(x.double(), w.double()),
                 lambda: ops.linear_f32_thirds(torch.randn(100, 66, device=DEV)[:, 1:65], w)):
        with pytest.raises((RuntimeError, ValueError, TypeError)):
            call()
