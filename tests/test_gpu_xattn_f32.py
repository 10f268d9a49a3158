"""The fp32 matrix attention (csrc/xattn_f32.hip) where its tiles end: row groups, key tiles, pages, chunks, kv splits, values that are
not numbers -- against the plain implementation (oracle/layered_ref.py) and the plain kernel, on the GPU (-m gpu)."""
import pytest
import torch

from oracle import layered_ref as lr
from tests.test_gpu_layers import BF, DEV, F32, Seqs, attention_case, ops  # noqa: F401

pytestmark = pytest.mark.gpu
# sums of up to 1 500 fp32 products and weights in any order: |error| <= n * 2^-24 * sum |terms|, far below this for such rows
TOL = 2e-5


@pytest.mark.parametrize("page", [32, 96, 128])
@pytest.mark.parametrize("H,KH,D,DV,chunk", [(4, 2, 64, 64, 0), (16, 1, 64, 40, 65), (6, 2, 100, 128, 64), (2, 2, 130, 200, 0)])
def test_row_and_key_edges(ops, H, KH, D, DV, chunk, page):  # noqa: F811
    """Portions that end just before, at and just behind a row group and a key tile; both kernels see the same cache."""
    lens = [300, 200]
    spec, rows, ref = attention_case(ops, H, KH, D, DV, chunk, H + D, F32, lens)
    for n0, n1 in ((1, 1), (4, 5), (15, 17), (16, 33), (31, 32), (63, 65), (64, 66), (127, 129)):
        s = Seqs(ops, spec, F32, lens, page=page, seed=n0)
        at = [lens[0] - n0 - n1, lens[1] - n1]
        s.attend(torch.cat([rows[b][:at[b]] for b in (0, 1)]), [0, 1], [0, 0], at)
        part = torch.cat([rows[0][at[0]:at[0] + n0], rows[1][at[1]:]])
        want = torch.cat([ref[0][at[0]:at[0] + n0], ref[1][at[1]:]])
        got = s.attend(part, [0, 1], at, [n0, n1])
        plain = s.attend(part, [0, 1], at, [n0, n1], plain=True)
        lim = TOL * max(1.0, float(want.abs().max()))
        assert float((got.double() - want).abs().max()) <= lim and float((got - plain).abs().max()) <= lim, (n0, n1)


@pytest.mark.parametrize("H,KH,D,DV,count", [(20, 4, 64, 64, 38), (20, 4, 128, 100, 38), (12, 4, 256, 256, 38), (20, 4, 64, 64, 35)])
def test_wide_row_groups(ops, H, KH, D, DV, count):  # noqa: F811
    """Many sequences of several rows: wide row groups from 144 of them on (the last case: 140), the last group and key tile of
    each sequence partly filled, a sequence of one key among them."""
    lens = [(17, 40, 64, 65, 90)[b % 5] for b in range(count)]
    spec, rows, ref = attention_case(ops, H, KH, D, DV, 0, D, F32, lens)
    s, who = Seqs(ops, spec, F32, lens, page=96, seed=2), list(range(count))
    at = [n - min(n, 1 + 4 * (b % 4)) for b, n in enumerate(lens)]
    at[3] = 0
    s.attend(torch.cat([r[:n] for r, n in zip(rows, at)]), who, [0] * count, at)
    part, new = torch.cat([r[n:] for r, n in zip(rows, at)]), [n - a for n, a in zip(lens, at)]
    want = torch.cat([r[n:] for r, n in zip(ref, at)])
    got, plain = (s.attend(part, who, at, new, plain=x) for x in (False, True))
    lim = TOL * max(1.0, float(want.abs().max()))
    assert float((got.double() - want).abs().max()) <= lim and float((got - plain).abs().max()) <= lim
    one = Seqs(ops, spec, F32, [1] * count, page=96, seed=3).attend(torch.cat([r[:1] for r in rows]), who, [0] * count, [1] * count)
    assert float((one.double() - torch.cat([r[:1] for r in ref])).abs().max()) <= lim


@pytest.mark.parametrize("H,KH,D", [(4, 1, 64), (32, 1, 128), (2, 2, 256)])
def test_kv_splits(ops, H, KH, D):  # noqa: F811
    """Few rows over many keys: the range is split over workgroups and merged, with and without a chunk that ends inside a split."""
    for chunk in (0, 1000):
        spec, rows, ref = attention_case(ops, H, KH, D, D, chunk, D, F32, [1500])
        s = Seqs(ops, spec, F32, [1500], seed=1)
        s.attend(rows[0][:1490], [0], [0], [1490])
        for n in (1, 2, 7):
            got = s.attend(rows[0][1490:1490 + n], [0], [1490], [n])
            assert float((got.double() - ref[0][1490:1490 + n]).abs().max()) <= TOL * max(1.0, float(ref[0].abs().max())), (chunk, n)


def test_a_value_that_is_no_number_reaches_only_rows_that_see_it(ops):  # noqa: F811
    for bad in (float("nan"), float("inf")):
        spec, rows, ref = attention_case(ops, 4, 2, 64, 64, 0, 3, F32, [150])
        v0 = (spec.H + spec.KH) * spec.D
        rows[0][70, v0:v0 + 64] = bad                       # kv head 0, position 70
        got = Seqs(ops, spec, F32, [150]).attend(rows[0], [0], [0], [150]).view(150, 4, 64)
        assert torch.isfinite(got[:70]).all() and torch.isfinite(got[:, 2:]).all()
        assert not torch.isfinite(got[70:, :2]).any()
        want = ref[0].view(150, 4, 64)
        assert float((got[:70].double() - want[:70]).abs().max()) <= TOL * float(want.abs().max())


@pytest.mark.parametrize("chunk", [0, 65])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_value_with_a_weight_of_zero(ops, bad, chunk):  # noqa: F811
    """Scores of up to 200 leave most weights at 0 in fp32: 0 times an infinity that a row sees is no number, as in the plain kernel --
    the same elements of both are numbers, over whole prompts and for a few rows (kv splits)."""
    for KH, D, n in ((2, 64, 300), (2, 64, 3), (1, 256, 300), (1, 128, 1)):
        spec, rows, _ = attention_case(ops, 4, KH, D, 64, chunk, 3, F32, [300], score=200.0)
        v0 = (spec.H + spec.KH) * spec.D
        rows[0][270, v0 + 5], rows[0][70, v0 + 9] = bad, -bad
        s = Seqs(ops, spec, F32, [300])
        s.attend(rows[0][:300 - n], [0], [0], [300 - n]) if n < 300 else None
        got, plain = (s.attend(rows[0][300 - n:], [0], [300 - n], [n], plain=x) for x in (False, True))
        assert torch.equal(torch.isfinite(got), torch.isfinite(plain)) and not torch.isfinite(plain).all()
        assert torch.allclose(got[torch.isfinite(plain)], plain[torch.isfinite(plain)], rtol=0, atol=TOL * 10)


def test_16_bit_pages_with_an_unknown_bound(ops):  # noqa: F811
    """Without a bound on the scores the bf16 kernels do not apply: same sums as the plain kernel, rounded once."""
    for H, KH, D, n in ((8, 2, 64, 100), (4, 4, 96, 5)):
        spec, rows, _ = attention_case(ops, H, KH, D, 64, 0, 5, BF, [120])
        spec.score_bound = 0.0
        s = Seqs(ops, spec, BF, [120])
        s.attend(rows[0][:120 - n], [0], [0], [120 - n])
        got, plain = (s.attend(rows[0][120 - n:], [0], [120 - n], [n], plain=x) for x in (False, True))
        assert torch.allclose(got.float(), plain.float(), rtol=2.0 ** -7, atol=1e-5)
