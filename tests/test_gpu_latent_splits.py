"""Decode steps of latent attention with few keys per workgroup: short and unequal sequences beside each other, splits of two to eight
tiles, some of them empty.  On the GPU (-m gpu)."""
import pytest
import torch

from tests.test_gpu_latent import BF, Seqs, attention_case, ops  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [[65], [129], [257], [300, 33], [700, 40, 130, 6], [200] * 13, [400, 90] * 9, [140] * 33])
@pytest.mark.parametrize("H,R,RD", [(16, 512, 64), (4, 64, 16), (40, 128, 32)])
def test_few_keys(ops, lens, H, R, RD):  # noqa: F811
    spec, zs, qs, gates, refs, _ = attention_case(ops, H, 32, RD, 32, 32, R, len(lens), BF, lens)
    s, who = Seqs(ops, spec, BF, lens, seed=2), list(range(len(lens)))
    before = [n - 3 for n in lens]
    s.attend(torch.cat([z[:n] for z, n in zip(zs, before)]), torch.cat([q[:n] for q, n in zip(qs, before)]), who, [0] * len(lens), before)
    for width, at in ((1, 0), (2, 1)):
        cut = [slice(n + at, n + at + width) for n in before]
        got, _ = s.attend(torch.cat([z[c] for z, c in zip(zs, cut)]), torch.cat([q[c] for q, c in zip(qs, cut)]), who,
                          [c.start for c in cut], [width] * len(lens), torch.cat([g[c] for g, c in zip(gates, cut)]))
        want = torch.cat([r[1][c] for r, c in zip(refs, cut)])
        assert float((got.double() - want).abs().max()) < 3e-2 * max(1.0, float(want.abs().max()))
