"""Host logic of the latent-attention decoder design without a GPU: weight loading, shared caches, the ragged step with its portions
and pages, the fixed-batch engine, the continuous-batching loop, over CPU stand-ins of the device ops that are built from the plain
implementation (they address pages the way the kernels do)."""
import pytest
import torch

from oracle import latent_ref as la
from oracle.layered_ref import rms
from tests import latent_util as lu
from tests.test_layers_cpu import _rows, resid_norm


def _pages(page_indices, page_indptr, b):
    return page_indices[int(page_indptr[b]):int(page_indptr[b + 1])].tolist()


def embed_bigram(tokens, table, pairs, norm_weight, eps, mul_before, mul_token, history, rows, page_indices, page_indptr):
    out = torch.empty(tokens.numel(), table.shape[1])
    page = history.shape[1]
    for b, r, n, pos in _rows(rows):
        pg = _pages(page_indices, page_indptr, b)
        before = int(history[pg[(pos - 1) // page], (pos - 1) % page]) if pos else None
        tk = tokens[r:r + n]
        out[r:r + n] = rms(table[tk] + pairs[la.bigram_rows(tk, before, mul_before, mul_token, pairs.shape[0] - 1)], eps) * norm_weight
        for j in range(n):
            history[pg[(pos + j) // page], (pos + j) % page] = int(tk[j])
    return out


class RotaryTable:
    def __init__(self, dims, base, max_pos, scaling=None, device=None):
        self.rot = {"dims": dims, "base": base}
        if scaling is not None:
            self.rot["scaling"] = dict(zip(("factor", "original", "fast", "slow"), scaling))
        self.max_pos, self.pairs = max_pos, dims // 2


def latent_append(z, s, cache, rows, page_indices, page_indptr, max_pages):
    if s.kv_norm is not None:
        for b, r, n, pos in _rows(rows):
            pg = _pages(page_indices, page_indptr, b)
            assert len(pg) * cache.shape[1] >= pos + n and len(pg) <= max_pages
            c, k = la.latent_keys(z[r:r + n, s.q_rank:s.q_rank + s.kv_rank + s.rot_dim], s.kv_norm, s.kv_rank, s.rotary.rot, s.eps, pos)
            for j in range(n):
                cache[pg[(pos + j) // cache.shape[1]], (pos + j) % cache.shape[1], :s.kv_rank + s.rot_dim] = torch.cat([c[j], k[j]])
    return rms(z[:, :s.q_rank], s.eps) * s.dq_norm


def latent_attention(q, s, cache, rows, page_indices, page_indptr, max_pages, workspace, out, gate=None, ctx=None):
    for b, r, n, pos in _rows(rows):
        if n == 0:
            continue
        pg = _pages(page_indices, page_indptr, b)
        held = torch.cat([cache[p] for p in pg])[:pos + n]
        o = la.latent_attention(q[r:r + n], held[:, :s.kv_rank], held[:, s.kv_rank:s.kv_rank + s.rot_dim], s.expand[:s.H * s.dim],
                                s.expand[s.H * s.dim:], s.H, s.dim, s.vdim, s.rotary.rot, s.scale, pos)
        out[r:r + n] = o * torch.sigmoid(gate[r:r + n]).unsqueeze(-1) if gate is not None else o
    if ctx is not None:
        assert ctx.new == [n for _, _, n, _ in _rows(rows)] and ctx.ctx == [pos + n for _, _, n, pos in _rows(rows)]
    return out


@pytest.fixture
def latent_ops(monkeypatch):
    from magicdec_amd import harness, ops
    for name, fn in (("embed_bigram", embed_bigram), ("resid_norm", resid_norm), ("RotaryTable", RotaryTable), ("latent_append", latent_append),
                     ("latent_attention", latent_attention), ("latent_row_width", lambda r, d: r + d + 3),
                     ("softcap_", la.softcap), ("argmax", lambda logits: logits.argmax(-1)), ("AttnWorkspace", lambda device: None),
                     ("gelu_mul", lambda a, b, out: out.copy_(la.gelu_tanh(a) * b))):
        monkeypatch.setattr(ops, name, fn)
    return harness


CFG = lu.config([lu.layer(2, heads=2, dim=10, rot_dim=6, vdim=12, q_rank=20, kv_rank=16, ff=40, yarn=lu.YARN), lu.layer(1, heads=3, mlp=False),
                 lu.layer(2, heads=5, dim=6, rot_dim=6, vdim=20, q_rank=14, kv_rank=16, ff=30, yarn=lu.YARN, kv_from=0)], vocab=90, width=48)


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    return lu.make(tmp_path_factory.mktemp("latent_cpu"), CFG, 3)


def engine(folder, slots, pages=None, max_len=300):
    from magicdec_amd.Engine.SnapKV.backend import LMBackend
    e = LMBackend(dtype=torch.float32, device="cpu")
    e.load_model(folder, use_tp=False)
    e.setup_caches(max_batch_size=slots, max_seq_length=max_len, num_pages=pages)
    for layer in e.model.layers:
        layer.attention.kv_cache.rows.fill_(float("nan"))
    e.model._history.fill_(17)
    return e


def test_layers_share_one_cache_and_the_head_is_the_embedding(latent_ops, model):
    e = engine(model[0], slots=2)
    a, b, c = (layer.attention for layer in e.model.layers)
    assert c.kv_cache is a.kv_cache and b.kv_cache is not a.kv_cache and c.kv_norm is None and c.cuts == [14, 0, 0]
    assert e.model.output.weight is e.model.tok_embeddings.weight and e.model._rowmajor_in_decode(e.model.output.weight)
    assert e.model._xspec[0].rotary is e.model._xspec[2].rotary and e.model.rollback_depth() is None


def test_the_product_in_fills_whole_tiles_of_columns(latent_ops, model):
    """32 columns each; the rows behind the parts are zeros, the parts where the checkpoint's are."""
    for layer in engine(model[0], slots=1).model.layers:
        att, n = layer.attention, sum(layer.attention.cuts)
        w = att.win.weight
        assert w.shape[0] % 32 == 0 and n <= w.shape[0] < n + 32 and not w[n:].any() and bool(w[:n].any(1).all())


@pytest.mark.parametrize("assign", [False, True])
def test_a_state_dict_without_the_rows_of_zeros_loads(latent_ops, model, assign):
    """One saved where the product in ended with the parts."""
    m = engine(model[0], slots=1).model
    whole = {k: v.clone() for k, v in m.state_dict().items()}
    saved = {k: v[:sum(m.layers[int(k.split(".")[1])].attention.cuts)].clone() if k.endswith("win.weight") else v.clone() for k, v in whole.items()}
    assert any(saved[k].shape != whole[k].shape for k in whole)
    for sd in (saved, whole):
        for p in m.parameters():
            p.data.fill_(7.0)
        m.load_state_dict(dict(sd), assign=assign)
        assert all(torch.equal(v, whole[k]) for k, v in m.state_dict().items())


@pytest.mark.parametrize("switch,value", [("set_mode", "lib"), ("set_mode", "hip"), ("set_fused", "0"), ("set_fused", "1"), (None, None)])
def test_the_switches_decide_where_a_steps_queries_run(latent_ops, model, monkeypatch, switch, value):
    """The query product shares a launch with the norm in front of it only where the policy is left to itself."""
    from magicdec_amd import ops
    from magicdec_amd.Engine import gemm_policy as g
    if g.mode() != "auto" or g.fused_mode() != "auto":
        pytest.skip("policy overridden by the environment")
    e, joint = engine(model[0], slots=1), []
    e.step([("a", [5, 6, 7])])

    def query(z, s, weight, cache, *where):
        joint.append(weight)
        return torch.nn.functional.linear(ops.latent_append(z, s, cache, *where), weight)
    monkeypatch.setattr(ops, "latent_query_supported", lambda *a: True)
    monkeypatch.setattr(ops, "latent_query", query)
    monkeypatch.setattr(e.model, "_gated_beside", lambda *a: None)
    e.model._packed.update({id(b.attention.wuq.weight): b.attention.wuq.weight for b in e.model.layers})
    if switch:
        old = {"set_mode": g.mode(), "set_fused": g.fused_mode()}[switch]
        getattr(g, switch)(value)
    try:
        e.step([("a", [8])])
    finally:
        if switch:
            getattr(g, switch)(old)
    assert len(joint) == (0 if switch else len(e.model.layers))


def test_copies_for_prompts_come_behind_those_for_steps(latent_ops, tmp_path, monkeypatch):
    """A card that holds the streaming copies that steps read, but not wukv's beside them, keeps the former; one rank of a group without
    room for wukv's is enough for none to make them."""
    from types import SimpleNamespace
    cfg = lu.config([lu.layer(2, heads=16, dim=48, rot_dim=64, vdim=64, q_rank=384, kv_rank=512, ff=512, yarn=lu.YARN)], vocab=512, width=512)
    lu.make(tmp_path / "m", cfg, 3)
    from magicdec_amd.Engine.SnapKV.backend import LMBackend
    e = LMBackend(dtype=torch.bfloat16, device="cpu")
    e.load_model(tmp_path / "m", use_tp=False)
    e.setup_caches(max_batch_size=1, max_seq_length=300)
    m, free = e.model, [1 << 40]
    monkeypatch.setattr(torch.cuda, "empty_cache", lambda: None)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda dev=None: (free[0], 1 << 40))

    def packed(room):
        free[0] = room + (6 << 30)
        m._pack_weights(force=True)
        return {m._roles[k][0] for k in m._packed}
    every = packed(1 << 40)
    size = lambda: sum(w.numel() * 2 for w in m._by_id.values())
    total, wukv = size(), m.layers[0].attention.wukv.weight.numel() * 2
    assert "wukv" in every and len(every) > 1
    assert packed(total) == every and packed(total - 1) == every - {"wukv"} == packed(total - wukv) and packed(total - wukv - 1) == set()
    dist = torch.distributed
    for name, fn in (("is_initialized", lambda: True), ("get_backend", lambda g: "gloo")):
        monkeypatch.setattr(dist, name, fn)
    m.replica_group = SimpleNamespace()
    for other, want in ((2, every), (1, every - {"wukv"}), (0, set())):
        monkeypatch.setattr(dist, "all_reduce", lambda t, op, group: t.clamp_(max=other))
        assert packed(total) == want


@pytest.mark.parametrize("portion_rows", [6, 17, 1000])
def test_ragged_steps_portions_and_reuse(latent_ops, model, monkeypatch, portion_rows):
    from magicdec_amd.Engine import backend_core
    monkeypatch.setattr(backend_core, "PREFILL_ROWS", portion_rows)
    folder, ref = model
    e = engine(folder, slots=3, pages=5)
    e.model.prefill_rows = portion_rows
    for trial in range(2):                              # the second time in slots and pages that were used
        seqs = {k: lu.tokens(n, 90, 10 * trial + n) for k, n in (("a", 140), ("b", 1), ("c", 41))}
        want = {k: ref.logits(v) for k, v in seqs.items()}
        cut = {"a": 133, "b": 1, "c": 22}
        toks, lg = e.step([(k, s[:cut[k]]) for k, s in seqs.items()], [list(range(cut[k])) for k in seqs])
        assert float(lu.row_errors(lg, torch.cat([want[k][:cut[k]] for k in seqs])).max()) < 1e-5
        assert toks.tolist() == [int(want[k][cut[k] - 1].argmax()) for k in seqs]
        e.end("b")
        for t in range(7):
            now = ("c", "a") if t % 2 else ("a", "c")
            _, lg = e.step([(k, seqs[k][cut[k] + t:cut[k] + t + 1]) for k in now], [[0], [0]], sample=False)
            assert float(lu.row_errors(lg, torch.stack([want[k][cut[k] + t] for k in now])).max()) < 1e-5
        e.end("a")
        _, lg = e.step([("c", seqs["c"][29:])], [[0, 11]], sample=False)      # a later portion of a prompt
        assert float(lu.row_errors(lg, want["c"][[29, 40]]).max()) < 1e-5
        e.end("c")
    assert sorted(e.pool.free_pages) == list(range(5)) and sorted(e.pool.free_slots) == [0, 1, 2]


def test_fixed_batch_generation(latent_ops, model):
    folder, ref = model
    e = engine(folder, slots=2, max_len=200)
    e.prefill_chunk = 32
    prompts = torch.tensor([lu.tokens(101, 90, s) for s in (1, 2)])
    out, steps, _ = latent_ops.run_baseline_batch(e, prompts, 140, -1, -1)
    for b in (0, 1):
        assert out[b, 101:].tolist() == ref.greedy(prompts[b].tolist(), 39)[0]


def test_continuous_batching(latent_ops, model):
    folder, ref = model
    e = engine(folder, slots=2, pages=3)
    prompts = [lu.tokens(n, 90, n) for n in (120, 3, 130, 1)]
    out, _, _ = latent_ops.run_sequences(e, prompts, 9)
    for p, o in zip(prompts, out):
        assert o == ref.greedy(p, 9)[0]


def test_weights_that_do_not_fit_the_config_are_refused(model, tmp_path):
    from magicdec_amd.Engine.SnapKV.backend import LMBackend
    t = lu.tensors(CFG, 1)
    for change, err in ((lambda d: d.pop("l1.mix.g"), KeyError), (lambda d: d.update({"l2.mix.dkv": d["l0.mix.dkv"].clone()}), KeyError),
                        (lambda d: d.update({"l0.mix.uk": d["l0.mix.uk"][:-1]}), ValueError), (lambda d: d.update(head=d["embed"].clone()), KeyError)):
        d = dict(t)
        change(d)
        folder = lu.write_model(tmp_path / "bad", CFG, d)
        with pytest.raises(err):
            LMBackend(dtype=torch.float32, device="cpu").load_model(folder, use_tp=False)
    with pytest.raises(NotImplementedError, match="tensor parallelism"):
        LMBackend(dtype=torch.float32, device="cpu").load_model(model[0], use_tp=True)


def test_named_configurations(tmp_path):
    from magicdec_amd.Engine import designs
    spec = designs.find_design(tmp_path / "Bufodra-8B" / "model.pth")
    assert spec.design == "Bufodra" and spec.dim == 4096 and spec.layers[3].attention.kv_from == 1
    assert [s.attention.kv_from for s in spec.layers[:8]] == [None, None, None, 1, None, None, None, 5]
