"""Driver entry points: build() compiles every HIP source for gfx950 (works without a GPU), smoke() runs one
tiny draft/verify iteration of the hot path on cuda:0 and checks it against the oracle."""
import math
import os
import sys

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def build() -> None:
    """hipcc --offload-arch=gfx950 for every kernel -> magicdec_amd/libmagicdec_hip.so (in-tree), then import the
    package and check that the library exports every symbol include/magicdec_hip.h declares."""
    from magicdec_amd.build_lib import build_library
    build_library(force=True)
    import magicdec_amd  # noqa: F401
    from magicdec_amd import _lib
    lib = _lib.load()
    assert lib.md_abi_version() == _lib.ABI_VERSION
    # the oracle is pure Python/numpy (the reference is Python): nothing to compile; oracle/_ref is not applicable
    # (the reference has no native sources)
    import oracle.flashinfer_ref  # noqa: F401
    import oracle.magicdec_ref  # noqa: F401
    print(f"[build] {_lib.LIB_PATH}: {len(_lib.EXPORTED_SYMBOLS)} C-ABI symbols OK")


def smoke() -> None:
    """One speculative iteration (3 StreamingLLM draft steps + 1 verify + fused accept) of a tiny GQA model on
    cuda:0 through the HIP library, checked against the CPU oracle (tokens tie-aware, page-table state exact)."""
    import tempfile

    import torch

    from magicdec_amd import _lib, harness
    from magicdec_amd.Engine import model_core
    from magicdec_amd.Engine.SnapKV.backend import LMBackend
    from magicdec_amd.Engine.StreamingLLM.backend_draft import LMBackend_Draft
    from oracle import magicdec_ref as mr

    _lib.load()
    assert torch.cuda.is_available(), "smoke() needs a GPU"
    dev = "cuda:0"
    cfg = mr.RefConfig(n_layer=2, n_head=8, n_local_heads=2, dim=512, intermediate_size=1024, vocab_size=2048,
                       rope_base=500000.0, scaling_factor=8, high_freq_factor=4, low_freq_factor=1,
                       original_max_position_embeddings=8192)
    sd = mr.init_state_dict(cfg, 11, wo_scale=0.1)
    d = tempfile.mkdtemp(prefix="md_smoke_")
    os.makedirs(os.path.join(d, "smoketiny"))
    torch.save(sd, os.path.join(d, "smoketiny", "model.pth"))
    model_core.transformer_configs["smoketiny"] = dict(
        block_size=4096, n_layer=2, n_head=8, n_local_heads=2, dim=512, intermediate_size=1024, vocab_size=2048,
        rope_base=500000.0, scaling_factor=8, high_freq_factor=4, low_freq_factor=1,
        original_max_position_embeddings=8192)
    from pathlib import Path
    ck = Path(d) / "smoketiny" / "model.pth"
    B, S, ML, G, BUD = 2, 288, 384, 3, 129
    g = torch.Generator().manual_seed(0)
    ids = torch.randint(4, 2048, (B, S), generator=g)
    ids[:, 0] = 1

    eng = LMBackend(dtype=torch.bfloat16, device=dev, dec_len=G + 1)
    eng.load_model(ck, use_tp=False)
    eng.setup_caches(max_batch_size=B, max_seq_length=ML)
    drf = LMBackend_Draft(dtype=torch.bfloat16, device=dev)
    drf.load_model(ck, use_tp=False)
    drf.setup_caches(max_batch_size=B, draft_budget=BUD)

    st = harness.new_state(B, G, ML + 1, dev, ids.to(dev))
    st.tokens_buffer[:, :1] = eng.encode(ids.to(dev))[:, -1:]
    drf.encode(ids.to(dev))
    terminal, nd = harness.longspec_iteration(eng, drf, st, G, 2, 0, S + 80, False)
    torch.cuda.synchronize()

    # oracle: the same iteration on the CPU (teacher-forced with the HIP draft tokens so that the verify pass sees
    # identical inputs even if a draft token flipped at a near-tie)
    o_t = mr.RefEngine("target", cfg, sd, B, ML)
    o_d = mr.RefEngine("stream_draft", cfg, sd, B, 0, BUD)
    t0 = o_t.encode(ids)[:, -1:]
    o_d.encode(ids)
    hip_first = st.output[:, S].cpu()
    assert torch.equal(hip_first, t0.view(-1)), f"prefill token: hip {hip_first.tolist()} oracle {t0.view(-1).tolist()}"
    an = st.accept_nums.cpu()
    assert int(an.min()) >= 1 and int(an.max()) <= G + 1
    assert eng.cachelens.cpu().tolist() == [S + int(a) for a in an], (eng.cachelens, an)
    assert drf.cachelens.cpu().tolist() == [BUD + min(int(a), G) for a in an]
    # what the HIP verify consumed: token 0 + the gamma draft tokens = output[S .. S+accept) ++ rejected tail; the
    # accepted prefix is what we can reconstruct exactly, so verify with the oracle on the first accept_nums rows
    tb = torch.zeros(B, G + 1, dtype=torch.long)
    tb[:, :1] = t0
    for i in range(G):
        tb[:, i + 1:i + 2] = o_d.inference(tb[:, i].view(-1, 1))
    tt = o_t.inference(tb)
    lg = o_t.model.last_logits.float()
    hip_lg = eng.model._last_logits.float().cpu().view(lg.shape)
    # rows whose inputs provably agree: position 0 of every request (input = the prefill token)
    err0 = (hip_lg[:, 0] - lg[:, 0]).abs().max().item()
    # the measured gate of tests/test_gpu_engine.py: no further from the oracle than twice the distance of a second
    # valid implementation of the same bf16 arithmetic (the oracle with float64-evaluated, once-rounded linears), plus
    # two bf16 ulps at the logit scale
    o_alt = mr.RefEngine("target", cfg, sd, B, ML)
    mr.LINEAR_MODE = "fp64"
    try:
        o_alt.encode(ids)
        o_alt.inference(tb)
    finally:
        mr.LINEAR_MODE = "fp32"
    err_alt = (o_alt.model.last_logits.float().view(lg.shape)[:, 0] - lg[:, 0]).abs().max().item()
    ulp = 2.0 ** (math.floor(math.log2(max(lg[:, 0].abs().max().item(), 2.0 ** -126))) - 7)
    gate = 2.0 * err_alt + 2.0 * ulp
    assert err0 <= gate, f"verify logits row 0 differ from the oracle by {err0} > gate {gate} (fp64-linear oracle: {err_alt})"
    print(f"[smoke] accept_nums={an.tolist()} terminal={terminal} next_double={nd} "
          f"max|verify logit diff row0| vs oracle={err0:.4f} (gate {gate:.4f} = 2 x {err_alt:.4f} + 2 ulp)")
    print("[smoke] OK")


if __name__ == "__main__":
    build()
    if len(sys.argv) > 1 and sys.argv[1] == "smoke":
        smoke()
