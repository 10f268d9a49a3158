"""md_linear_prompt (csrc/promptgemm.hip) against float64 products, at the edges of its tiles.  On the GPU (-m gpu)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TILES = (0, 256256, 192256, 128256, 256128, 192128, 128128)


def case(M, N, K, seed, ldx=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K + ldx, device=DEV, generator=g).bfloat16()[:, :K]
    return x, (torch.randn(N, K, device=DEV, generator=g) * 0.1).bfloat16(), torch.randn(N, device=DEV, generator=g).bfloat16()


def product(x, w):
    """(float64 product, bound on what fp32 sums of K terms are off it)"""
    return x.double() @ w.double().t(), (x.double().abs() @ w.double().abs().t()) * (x.shape[1] * 2.0 ** -24)


U = 2.0 ** -8            # half an ulp of bf16 relative to the value: 8 significant bits, the spacing in [1, 2) is 2^-7


# rows and columns around a tile's and a wavefront's edge, one row, one piece of 8 columns, several tiles per workgroup, K of 4, 8 and 12 steps
@pytest.mark.parametrize("M,N,K,ldx", [(1, 8, 256, 0), (257, 264, 256, 8), (300, 520, 512, 0), (127, 1000, 768, 64), (769, 96, 512, 0),
                                       (2049, 1032, 256, 0), (1000, 20000, 256, 0)])
def test_products(M, N, K, ldx):
    from magicdec_amd import ops
    x, w, bias = case(M, N, K, M, ldx)
    ref, off = product(x, w)
    plain = ops.PackedWeight(w)
    first = None
    for tile in TILES:
        wide = torch.full((M + 1, N + 16), -7.0, device=DEV, dtype=torch.bfloat16)
        out = ops.linear_prompt(x, plain, out=wide[:M, 8:8 + N], tile=tile)
        assert ((out.double() - ref).abs() <= ref.abs() * U + 2 * off).all()
        assert (wide[M] == -7).all() and (wide[:, :8] == -7).all() and (wide[:, 8 + N:] == -7).all()       # nothing beside it
        first = out.clone() if first is None else first
        assert torch.equal(out, first)                                                                    # the same bits from every tile
        got = ops.linear_prompt(x, plain, bias, tile=tile)
        want = ref + bias.double()
        assert ((got.double() - want).abs() <= want.abs() * U + 2 * off + 2.0 ** -23 * bias.double().abs()).all()


@pytest.mark.parametrize("M,N,K", [(257, 272, 256), (129, 2000, 512), (1025, 1040, 512), (2100, 12000, 256)])
def test_activations(M, N, K):
    from magicdec_amd import ops
    x, w, _ = case(M, N, K, N)
    ref, off = product(x, w)
    act = torch.tensor([0.3, -0.2], device=DEV)
    a, b = torch.nn.functional.softplus(act.double())
    low = ref.clamp(max=0)
    z = ref / 2 + torch.where(ref > 0, a * ref * ref, (0.5 + b) * (torch.expm1(low) - low))
    slope = 0.5 + torch.where(ref > 0, 2 * a * ref, (0.5 + b) * (torch.exp(low) - 1).abs())
    h1, h3, o1, o3 = ref[:, :N // 2], ref[:, N // 2:], off[:, :N // 2], off[:, N // 2:]
    s = torch.sigmoid(h1)
    silu, dsilu = h1 * s, (s * (1 + h1 * (1 - s))).abs()
    gelu = torch.nn.functional.gelu(h1, approximate="tanh")
    for tile in TILES:
        got = ops.linear_prompt(x, ops.PackedWeight(w), xielu=act, tile=tile).double()
        # (the exponential's argument and result: 2 ulp of float)
        assert ((got - z).abs() <= z.abs() * U + slope * 2 * off + 2.0 ** -22 * (1 + ref.abs())).all()
        gated = ops.PackedWeight(w, swiglu=True)
        got = ops.linear_prompt(x, gated, swiglu=True, tile=tile).double()
        # rounded: h1, h3, silu(h1), the product
        bound = (dsilu * (h1.abs() * U + 2 * o1) * h3.abs() + silu.abs() * 2 * o3 + 3 * U * (silu * h3).abs()) * 1.02 + 1e-30
        assert ((got - silu * h3).abs() <= bound).all()
        got = ops.linear_prompt(x, gated, swiglu=True, gelu=True, tile=tile).double()
        bound = 1.13 * 2 * o1 * h3.abs() + gelu.abs() * 2 * o3 + U * (gelu * h3).abs() + 2.0 ** -20 * (1 + h1.abs()) * h3.abs()
        assert ((got - gelu * h3).abs() <= bound).all()


def test_silu_of_every_number_is_a_steps():
    """SiLU of all finite bf16 numbers (a product with the identity) has the bits of the kernel beside the library's products."""
    from magicdec_amd import ops
    h1 = torch.arange(65536, dtype=torch.int32, device=DEV).to(torch.int16).view(torch.bfloat16).view(256, 256)
    h1 = torch.where(h1.abs() < 3e38, h1, 0)
    h1 = torch.where(h1.abs() > 1e-36, h1, 0)                                 # (no products that are not normal numbers)
    eye = torch.eye(256, device=DEV).bfloat16()
    for big in (1.0, 2.0 ** 100):                                             # ... of h1 from -88.5 on the SiLU is 1e-37
        h3 = torch.full_like(h1, big)
        want = ops.silu_mul(h1.t().contiguous(), h3)
        got = ops.linear_prompt(eye, ops.PackedWeight(torch.cat([h1, h3]), swiglu=True), swiglu=True)
        assert torch.equal(got, want)
        assert (want[(h1.t() >= -88.5) & (h1.t() < -87.4)] < -1e-37).all()


def test_activations_are_as_exact_as_a_steps():
    """xIELU and GELU of 32-bit sums, almost all of them the float64 value rounded once: a relative error e rounds the other way in a share
    e / 2^-9 at most.  xIELU has 1e-7 of its terms, GELU 2e-7 (behind -0.5 3e-6 and behind -2 1.3e-5, of its exponent); GELU twice that."""
    from magicdec_amd import ops
    g = torch.Generator(device=DEV).manual_seed(11)
    rows = torch.zeros(128, 256, device=DEV).bfloat16()
    rows[torch.arange(128), torch.arange(128) * 2] = rows[torch.arange(128), torch.arange(128) * 2 + 1] = 1
    N = 4096
    for lo, hi in ((-0.02, -0.0039), (-0.0039, -1e-3), (-0.1, -0.02), (-2.0, -0.1), (-9.9, -2.0), (0.01, 6.0)):
        grid = 2.0 ** (math.ceil(math.log2(max(-lo, hi))) - 16)               # of 16 bits: a sum of two numbers
        z = ((torch.rand(N, 128, device=DEV, generator=g) * (hi - lo) + lo) / grid).round() * grid
        top = z.bfloat16()
        low = (z - top.float()).bfloat16()
        w = torch.stack([top, low], 2).flatten(1)
        assert torch.equal(top.double() + low.double(), z.double())
        z = z.double().t()
        for av, bv in ((0.3, -0.2), (5.0, 5.0)):
            act = torch.tensor([av, bv], device=DEV)
            a, b = torch.nn.functional.softplus(act.double())
            want = z / 2 + torch.where(z > 0, a * z * z, (0.5 + b) * (torch.expm1(z.clamp(max=0)) - z))
            # (its terms may cancel: as much more as they are larger than their sum)
            share = 1e-7 * 512 * float((((0.5 + b) * z.clamp(max=0).abs() + z.abs() + a * z.clamp(min=0) ** 2) / want.abs().clamp(min=1e-4)).mean())
            got = ops.linear_prompt(rows, ops.PackedWeight(w), xielu=act)
            assert float((got != want.bfloat16()).float().mean()) <= share, (lo, av, share)
        ones = torch.zeros(N, 256, device=DEV).bfloat16()
        ones[:, ::2] = 1
        got = ops.linear_prompt(rows, ops.PackedWeight(torch.cat([w, ones]), swiglu=True), swiglu=True, gelu=True)
        want = z * torch.sigmoid(2 * math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3))
        assert float((got != want.bfloat16()).float().mean()) <= 2 * 512 * (1.3e-5 if lo < -2 else 3e-6 if lo < -0.5 else 2e-7), lo


def test_not_finite():
    """An infinity or NaN of a row stays in it; a saturated activation is 0 or its argument."""
    from magicdec_amd import ops
    x, w, _ = case(300, 64, 256, 3)
    x[7, 5], x[200, 100] = float("inf"), float("nan")
    for kw in ({}, dict(xielu=torch.tensor([0.3, -0.2], device=DEV)), dict(swiglu=True), dict(swiglu=True, gelu=True)):
        out = ops.linear_prompt(x, ops.PackedWeight(w, swiglu="swiglu" in kw), **kw)
        bad = ~torch.isfinite(out).all(1)
        assert bad[7] and bad[200] and bad.sum() == 2 and out[200].isnan().all()
    big = torch.full((300, 256), 1.0, device=DEV).bfloat16()
    w = torch.cat([torch.full((8, 256), -1.0), torch.full((8, 256), 1.0), torch.full((16, 256), 0.5)]).to(DEV).bfloat16()     # h1 = -256, 256
    for gelu in (False, True):
        out = ops.linear_prompt(big, ops.PackedWeight(w, swiglu=True), swiglu=True, gelu=gelu)
        assert (out[:, :8] == 0).all() and (out[:, 8:] == 256 * 128).all()


def test_refused():
    from magicdec_amd import ops
    x, w, bias = case(300, 64, 256, 5)
    pw = ops.PackedWeight(w)
    for call in (lambda: ops.linear_prompt(x[:, :128], ops.PackedWeight(w[:, :128].contiguous())),            # K: no multiple of 256
                 lambda: ops.linear_prompt(x, ops.PackedWeight(w[:60].contiguous())),                       # columns: no multiple of 8
                 lambda: ops.linear_prompt(x, pw, tile=64064),
                 lambda: ops.linear_prompt(x, pw, bias[:32]),
                 lambda: ops.linear_prompt(x, pw, out=torch.empty(300, 68, device=DEV, dtype=torch.bfloat16)[:, 2:66])):       # alignment
        with pytest.raises((RuntimeError, ValueError)):
            call()


@pytest.mark.parametrize("M,N,K,swiglu", [(4112, 4096, 5120, False), (8193, 2048, 2560, False), (4224, 4096, 9216, False), (10241, 16384, 2048, True)])
def test_rows_behind_whole_tiles(M, N, K, swiglu):
    """A linear of a prompt whose last rows run on the weight-streaming kernel: every row against float64, in a view of a wider matrix."""
    from types import SimpleNamespace
    from magicdec_amd import ops
    from magicdec_amd.Engine.gemm_policy import prompt_rows
    from magicdec_amd.Engine.model_core import Transformer
    assert 0 < prompt_rows(M, N, K, swiglu) < M
    x, w, bias = case(M, N, K, M)
    pk, n_out = ops.PackedWeight(w, swiglu=swiglu), N // 2 if swiglu else N
    model = SimpleNamespace(workspace=ops.AttnWorkspace(DEV))
    wide = torch.full((M, n_out + 8), -7.0, device=DEV, dtype=torch.bfloat16)
    out = Transformer._prompt_linear(model, x, pk, None if swiglu else bias, swiglu, out=wide[:, :n_out])
    assert (wide[:, n_out:] == -7).all() and out.data_ptr() == wide.data_ptr()
    ref, off = product(x, w)
    if not swiglu:
        want = ref + bias.double()
        assert ((out.double() - want).abs() <= want.abs() * U + 2 * off + 2.0 ** -23 * bias.double().abs()).all()
        return
    h1, h3 = ref[:, :n_out], ref[:, n_out:]
    s = torch.sigmoid(h1)
    bound = ((s * (1 + h1 * (1 - s))).abs() * (h1.abs() * U + 2 * off[:, :n_out]) * h3.abs() + (h1 * s).abs() * 2 * off[:, n_out:]
             + 3 * U * (h1 * s * h3).abs()) * 1.02 + 1e-30
    assert ((out.double() - h1 * s * h3).abs() <= bound).all()


@pytest.mark.parametrize("M,N,K,kind", [(4112, 4096, 5120, "xielu"), (8193, 2048, 2560, "xielu"), (10241, 16384, 2048, "gelu"), (10241, 16384, 2048, "swiglu")])
def test_activations_of_rows_behind_whole_tiles(M, N, K, kind):
    """The same with the activations, into columns of a wider matrix: both kernels' rows against float64, nothing beside them."""
    from types import SimpleNamespace
    from magicdec_amd import ops
    from magicdec_amd.Engine.gemm_policy import prompt_rows
    from magicdec_amd.Engine.model_core import Transformer
    gated = kind != "xielu"
    rows = prompt_rows(M, N, K, gated)
    assert 0 < rows < M
    x, w, _ = case(M, N, K, M + 1)
    act = torch.tensor([0.3, -0.2], device=DEV)
    n_out = N // 2 if gated else N
    wide = torch.full((M, n_out + 24), -7.0, device=DEV, dtype=torch.bfloat16)
    kw = dict(xielu=act) if not gated else dict(gelu=True) if kind == "gelu" else {}
    out = Transformer._prompt_linear(SimpleNamespace(workspace=ops.AttnWorkspace(DEV)), x, ops.PackedWeight(w, swiglu=gated), None, gated,
                                     out=wide[:, 16:16 + n_out], **kw)
    assert (wide[:, :16] == -7).all() and (wide[:, 16 + n_out:] == -7).all() and out.data_ptr() == wide[:, 16:].data_ptr()
    for lo in range(0, M, 2048):                                              # (in parts: float64 of all rows is much)
        part, got = x[lo:lo + 2048], out[lo:lo + 2048].double()
        ref, off = product(part, w)
        if kind == "xielu":
            a, b = torch.nn.functional.softplus(act.double())
            low = ref.clamp(max=0)
            z = ref / 2 + torch.where(ref > 0, a * ref * ref, (0.5 + b) * (torch.expm1(low) - low))
            slope = 0.5 + torch.where(ref > 0, 2 * a * ref, (0.5 + b) * (torch.exp(low) - 1).abs())
            assert ((got - z).abs() <= z.abs() * U + slope * 2 * off + 2.0 ** -22 * (1 + ref.abs())).all()
            continue
        h1, h3, o1, o3 = ref[:, :n_out], ref[:, n_out:], off[:, :n_out], off[:, n_out:]
        if kind == "gelu":
            gelu = torch.nn.functional.gelu(h1, approximate="tanh")
            bound = 1.13 * 2 * o1 * h3.abs() + gelu.abs() * 2 * o3 + U * (gelu * h3).abs() + 2.0 ** -20 * (1 + h1.abs()) * h3.abs()
            assert ((got - gelu * h3).abs() <= bound).all()
        else:
            s = torch.sigmoid(h1)
            bound = ((s * (1 + h1 * (1 - s))).abs() * (h1.abs() * U + 2 * o1) * h3.abs() + (h1 * s).abs() * 2 * o3 + 3 * U * (h1 * s * h3).abs()) * 1.02 + 1e-30
            assert ((got - h1 * s * h3).abs() <= bound).all()


@pytest.mark.parametrize("M,N,K,swiglu,taken", [(129, 33024, 512, True, True), (192, 65536, 256, False, True), (256, 37888, 512, True, True),
                                                (256, 32768, 512, True, False), (128, 37888, 512, True, False), (255, 152064, 256, False, False)])
def test_a_steps_rows_in_the_place_of_the_block_kernel(M, N, K, swiglu, taken, monkeypatch):
    """Both sides of the rule's lines, through the model's linear; every row against float64."""
    from types import SimpleNamespace
    from magicdec_amd import ops
    from magicdec_amd.Engine import gemm_policy
    from magicdec_amd.Engine.model_core import Transformer
    monkeypatch.setattr(gemm_policy, "choose", lambda *a, **kw: "block")
    x, w, bias = case(M, N, K, M)
    assert gemm_policy.prompt_over_block(M, N, K, swiglu) == taken
    calls, real = [], ops.linear_prompt
    monkeypatch.setattr(ops, "linear_prompt", lambda *a, **kw: calls.append(1) or real(*a, **kw))
    pk = ops.PackedWeight(w, swiglu=swiglu)
    model = SimpleNamespace(workspace=ops.AttnWorkspace(DEV), _packed={id(w): pk}, _on_prompt_gemm=Transformer._on_prompt_gemm)
    model._prompt_linear = lambda *a, **kw: Transformer._prompt_linear(model, *a, **kw)
    out = Transformer._linear(model, x, SimpleNamespace(weight=w, bias=None if swiglu else bias), swiglu_w13=(w, None) if swiglu else None)
    assert len(calls) == taken
    ref, off = product(x, w)
    if swiglu:
        h1, h3 = ref[:, :N // 2], ref[:, N // 2:]
        s = torch.sigmoid(h1)
        # (the block kernel rounds both halves and the SiLU to bf16: as many half-ulps as roundings)
        bound = ((s * (1 + h1 * (1 - s))).abs() * (h1.abs() * U + 2 * off[:, :N // 2]) * h3.abs() + (h1 * s).abs() * 2 * off[:, N // 2:]
                 + 3 * U * (h1 * s * h3).abs()) * 1.02 + 1e-30
        assert ((out.double() - h1 * s * h3).abs() <= bound).all()
    else:
        want = ref + bias.double()
        assert ((out.double() - want).abs() <= want.abs() * U + 2 * off + 2.0 ** -23 * bias.double().abs()).all()


def test_a_step_of_more_than_256_rows_reads_one_copy_of_its_weights(monkeypatch):
    """After a prompt the weights that such steps multiply on md_linear_prompt have their streaming copy only, and the step asks for no
    other: the logits have the bits of an engine that keeps both."""
    from pathlib import Path
    from magicdec_amd.Engine import model_core
    from magicdec_amd.Engine.SnapKV.backend import LMBackend
    monkeypatch.setitem(model_core.transformer_configs, "one-copy", dict(block_size=512, n_layer=2, vocab_size=4096, n_head=16, n_local_heads=4, dim=2048,
                                                                         intermediate_size=8192))
    B, n, got = 65, 6, []
    ids = torch.randint(0, 4096, (B, 140), generator=torch.Generator().manual_seed(0)).to(DEV)
    for keep in ("0", "1"):
        monkeypatch.setenv("MAGICDEC_KEEP_ROWMAJOR", keep)
        e = LMBackend(dtype=torch.bfloat16, device=DEV, dec_len=n)
        torch.manual_seed(1)
        e.load_model(Path("no-checkpoint/one-copy/model.pth"), use_tp=False)
        e.setup_caches(max_batch_size=B, max_seq_length=256)
        e.encode(ids)
        e.inference(ids[:, :n])
        got.append((e.model._last_logits.clone(), getattr(e.model, "_warned_transient", False), len(e.model._released)))
    assert torch.equal(got[0][0], got[1][0]) and not got[0][1] and got[0][2] > 0 == got[1][2]
