"""The integer work around a captured decode step (md_step_ops): every kind of piece alone and together, and a step whose length
tensors the caller replaces between replays.  On the GPU (-m gpu)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n", [1, 3, 255, 256, 257, 5000])
def test_pieces(n):
    from magicdec_amd import ops
    g = torch.Generator().manual_seed(n)
    a, b, src = (torch.randint(-1000, 1000, (n,), dtype=torch.int32, generator=g) for _ in range(3))
    wide = torch.randint(0, 1 << 40, (n, 5), generator=g)
    da, db, dst, out = a.to(DEV), b.to(DEV), torch.zeros(n, dtype=torch.int32, device=DEV), torch.zeros(n, 1, dtype=torch.int64, device=DEV)
    pair, dense = torch.zeros(n, 2, dtype=torch.int64, device=DEV), torch.zeros(n, 5, dtype=torch.int64, device=DEV)
    dw = wide.to(DEV)
    pieces = ops.StepOps(add=[(da, 4), (db, -7)], scale=[(dst, src.to(DEV), 3)], copies=[torch.zeros_like(out), pair, dense])
    pieces.run(dw[:, 3].view(-1, 1), dw[:, 1:3], dw, into=(out, pair, dense))
    assert torch.equal(da.cpu(), a + 4) and torch.equal(db.cpu(), b - 7) and torch.equal(dst.cpu(), src * 3)
    assert torch.equal(out.cpu(), wide[:, 3:4]) and torch.equal(pair.cpu(), wide[:, 1:3]) and torch.equal(dense.cpu(), wide)


@pytest.mark.parametrize("rows,cols", [(1, 1), (2, 255), (64, 126), (257, 1), (1, 300)])
def test_fills_and_grids(rows, cols):
    """Constants and page tables: every piece of a launch of eight, and what another launch takes."""
    from magicdec_amd import ops
    from magicdec_amd.Engine.backend_core import _Integers
    ints, want = _Integers(), []
    for k in range(5):
        t, u = (torch.full((rows * cols + 2,), -1, dtype=torch.int32, device=DEV)[1:-1] for _ in range(2))      # (views: nothing beside them)
        ints.fill(t, 7 - k)
        ints.grid(u, rows, cols + k)
        want += [(t, torch.full((rows, cols), 7 - k)), (u, torch.arange(rows).view(-1, 1) * (cols + k) + torch.arange(cols))]
    strided, src = torch.zeros(rows, 2, dtype=torch.int32, device=DEV)[:, 0], torch.arange(rows, dtype=torch.int32, device=DEV)
    ints.scale(strided, src, 3)                              # (not dense: torch writes it)
    ints.run()
    for t, w in want + [(strided, src.cpu() * 3)]:
        assert torch.equal(t.cpu(), w.int().view(t.shape))
    assert all(t._base[0].item() == -1 and t._base[-1].item() == -1 for t, _ in want)
    with pytest.raises(ValueError):
        ops.StepOps(grid=[(torch.zeros(5, dtype=torch.int32, device=DEV), 2, 1)])


def test_what_it_does_not_take():
    from magicdec_amd import ops
    t = torch.zeros(8, 2, dtype=torch.int64, device=DEV)
    i = torch.zeros(8, dtype=torch.int32, device=DEV)
    assert not ops.step_copies(t.int()) and not ops.step_copies(t.t()) and not ops.step_copies(t.cpu()) and not ops.step_copies(t[:0])
    assert ops.step_copies(t) and ops.step_copies(t[:, 1:]) and ops.step_adds(i) and not ops.step_adds(i[::2]) and not ops.step_adds(i.long())
    for bad in (dict(add=[(i, 1)] * 9), dict(add=[(i[::2], 1)]), dict(copies=[t.t()]), dict(scale=[(i, i[:4], 2)]), dict(copies=[i])):
        with pytest.raises(ValueError):
            ops.StepOps(**bad)
    with pytest.raises(TypeError):
        ops.StepOps(add=[(t, 1)])
    for src in (t.t(), t[:4], t.cpu(), t.int()):
        with pytest.raises(ValueError):
            ops.StepOps(copies=[t]).run(src)
    with pytest.raises(ValueError):
        ops.StepOps(copies=[t]).run()


def test_lengths_of_a_captured_step():
    """Tokens and lengths of captured steps equal the eager ones when length tensors are moved in place, replaced by tensors of the
    caller's, and put back (benchmark=True), on ids that are dense, a strided column and 32-bit."""
    from magicdec_amd.Engine.model_core import transformer_configs
    from magicdec_amd.Engine.SnapKV.backend import LMBackend
    transformer_configs["step-ops-test"] = dict(block_size=512, n_layer=1, n_head=2, n_local_heads=1, dim=128, intermediate_size=256, vocab_size=64)
    made = []
    for graphs in (False, True):
        e = LMBackend(dtype=torch.bfloat16, device=DEV)
        e.load_model("none/step-ops-test/model.pth", use_tp=False)
        if graphs:
            e.compile()
        e.setup_caches(max_batch_size=3, max_seq_length=256)
        g = torch.Generator().manual_seed(0)
        e.encode(torch.randint(4, 64, (3, 40), generator=g).to(DEV))
        got = []
        for k in range(8):
            ids = torch.randint(4, 64, (3, 5), generator=g).to(DEV)
            ids = ids[:, 2].view(-1, 1) if k % 3 == 0 else ids[:, :1].contiguous() if k % 3 == 1 else ids[:, 1].contiguous().view(-1, 1).int()
            if k == 3:
                e.cachelens, e.paged_kv_last_page_len = e.cachelens - 1, e.paged_kv_last_page_len - 1
            got += [e.inference(ids, benchmark=k == 5).cpu(), e.cachelens.cpu().clone(), e.paged_kv_last_page_len.cpu().clone()]
        made.append(got)
    assert all(torch.equal(a, b) for a, b in zip(*made))


@pytest.mark.parametrize("kinds", [(torch.int32,) * 3, (torch.int32, torch.int64, torch.int32), (torch.int64, torch.int32, torch.int64)])
def test_token_ids_of_either_width(kinds):
    """A step captured on 32-bit ids, and one that meets the other width later: tokens and lengths of the eager engine."""
    from magicdec_amd.Engine.model_core import transformer_configs
    from magicdec_amd.Engine.SnapKV.backend import LMBackend
    transformer_configs["step-ops-test"] = dict(block_size=512, n_layer=1, n_head=2, n_local_heads=1, dim=128, intermediate_size=256, vocab_size=64)
    made = []
    for graphs in (False, True):
        e = LMBackend(dtype=torch.bfloat16, device=DEV)
        e.load_model("none/step-ops-test/model.pth", use_tp=False)
        if graphs:
            e.compile()
        e.setup_caches(max_batch_size=3, max_seq_length=256)
        g = torch.Generator().manual_seed(1)
        e.encode(torch.randint(4, 64, (3, 40), generator=g).to(DEV))
        got = []
        for kind in kinds:
            got += [e.inference(torch.randint(4, 64, (3, 1), generator=g).to(kind).to(DEV)).cpu(), e.cachelens.cpu().clone(),
                    e.paged_kv_last_page_len.cpu().clone()]
        made.append(got)
        assert e._use_graphs == graphs                       # (no fall-back to eager steps)
    assert all(torch.equal(a, b) for a, b in zip(*made))


def test_uploads_behind_queued_work():
    """Many uploads back to back, while the stream still has work in front of them and their host memory is used again: every value; from
    lists, host tensors of either type, and tensors that are on the device already."""
    from magicdec_amd import ops
    a = torch.randn(4096, 4096, device=DEV)
    got = []
    for i in range(200):
        if i % 20 == 0:
            a = (a @ a).clamp_(-1, 1)
        n = 1 + 37 * i % 1000
        v = torch.arange(i, i + n, dtype=torch.long if i % 3 else torch.int32)
        v = v.pin_memory() if i % 4 == 3 else v
        src = v.tolist() if i % 4 == 0 else v.to(DEV) if i % 4 == 1 else v
        dtype = torch.int32 if i % 2 else torch.long
        got.append((i, n, dtype, ops.upload(src, dtype, DEV)))
        if i % 4 > 1:
            v.fill_(-1)                                        # the caller's tensor is its own again
    for i, n, dtype, t in got:
        assert t.dtype == dtype and t.is_cuda and torch.equal(t.cpu(), torch.arange(i, i + n, dtype=dtype)), i
