"""The work this framework is used for, as a list of measurable cases: what a serving or benchmark program asks of its engines, from one
short request to a batch of long ones.

A case runs a few layers of a model of the zoo (full width, 32 000 tokens) through the engine classes.  Weights, prompts and cache
contents come from the seed; where a step runs over a long context, the context's cache rows are drawn instead of computed.  The head
answers to the embedding of one other token per token, so that next-token distributions are as decided as a trained model's.

kinds:
    decode    one step of `rows` tokens per request over the full cache: autoregressive (1) or verification of a draft (gamma + 1)
    draft     one step of the stand-alone draft model over its SnapKV cache (2 rows: the step behind an all-accepted iteration)
    encode    prompts of equal length through the target engine
    stream    prompts through the StreamingLLM draft: a sink and a window, evicted portion by portion
    select    the compression of one layer's cache into the SnapKV draft cache
    prompts   prompts of equal length through a layered design
    steps     one decode step of a layered design behind its prompts
    ragged    continuous batching: prompts of unequal lengths, some decode steps, the sequences end
"""
import math

import torch

VOCAB = 32000
PAGE = 128
WINDOW, SINK, CHUNK = 32, 16, 128
FP8_SCALE = 6.0 / 448.0
DEV = "cuda:0"


def listed():
    return [
        # the smallest model's greedy step for one short request: launches and latency
        dict(name="68m-decode-b1", kind="decode", model="68m", layers=2, batch=1, context=129, rows=1, kv="bf16"),
        # one request with a long document on an 8B model
        dict(name="8b-decode-b1-32k", kind="decode", model="llama-3.1-8b", layers=2, batch=1, context=32064, rows=1, kv="bf16"),
        # verification of three draft tokens for a full batch of 16K contexts: the headline benchmark's target step
        dict(name="8b-verify-b64-16k", kind="decode", model="llama-3.1-8b", layers=1, batch=64, context=16032, rows=4, kv="bf16"),
        # the same for a model with five query heads per kv head, query / key / value biases and an fp8 cache
        dict(name="32b-verify-b32-fp8", kind="decode", model="Qwen2.5-32b", layers=1, batch=32, context=8096, rows=4, kv="fp8"),
        # the headline benchmark's draft step
        dict(name="1b-draft-b64", kind="draft", model="llama-3.2-1b", layers=4, batch=64, budget=257, context=4000, rows=1),
        # prompts of a few requests on the target
        dict(name="8b-encode-b4-2k", kind="encode", model="llama-3.1-8b", layers=2, batch=4, prompt=2081),
        # the same prompts' pass through a StreamingLLM draft
        dict(name="1b-stream-b16-2k", kind="stream", model="llama-3.2-1b", layers=4, batch=16, budget=257, prompt=2081),
        # what the SnapKV draft does with every layer of a long prompt
        dict(name="1b-select-b16-16k", kind="select", model="llama-3.2-1b", batch=16, budget=257, context=16032),
        # prompts of a layered design with chunked attention
        dict(name="furitar-prompts-b8-2k", kind="prompts", model="furitar-8b", layers=2, batch=8, prompt=2049, dtype="bf16"),
        # prompts and decode steps of a layered design with latent attention
        dict(name="bufodra-prompts-b4-2k", kind="prompts", model="bufodra-8b", layers=4, batch=4, prompt=2049, dtype="bf16"),
        dict(name="bufodra-steps-b32-2k", kind="steps", model="bufodra-1b", layers=4, batch=32, prompt=2049, dtype="bf16"),
        # a recorded trace of unequal requests replayed in 32-bit, as a design's results are checked
        dict(name="furitar-ragged-f32", kind="ragged", model="furitar-1b", layers=2, batch=6, shortest=100, longest=1500, steps=8,
             dtype="float32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _room(context, rows):
    """The nearest context whose last page has room for `rows` more tokens (what the fixed-batch engines ask for)."""
    return context - max(0, (context - 1) % PAGE + 1 + rows - PAGE)


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "draft", "encode", "stream", "select", "prompts", "prompts", "steps", "steps", "ragged"])
    if kind == "decode":
        model = rng.choice(["68m", "llama-3.2-1b", "llama-3.1-8b", "Qwen2.5-7b", "Qwen2.5-32b"])
        batch, rows = _log(rng, 1, 64), rng.choice([1, 1, 2, 4, 4, 6])
        context = _log(rng, 100, min(32000, 1000000 // batch) if model != "68m" else 1900)
        return dict(kind=kind, model=model, layers=2 if batch * context < 400000 else 1, batch=batch, context=_room(context, rows),
                    rows=rows, kv="bf16" if model == "68m" else rng.choice(["bf16", "bf16", "fp8"]))
    if kind == "draft":
        return dict(kind=kind, model=rng.choice(["llama-3.2-1b", "tinyllama"]), layers=4, batch=_log(rng, 1, 64),
                    budget=rng.choice([129, 257, 513]), context=rng.randrange(600, 2000), rows=rng.choice([1, 1, 2]))
    if kind == "encode":
        model, batch = rng.choice(["llama-3.2-1b", "llama-3.1-8b", "Qwen2.5-7b"]), _log(rng, 1, 8)
        return dict(kind=kind, model=model, layers=2, batch=batch, prompt=_log(rng, 65, 8000 // batch))
    if kind == "stream":
        batch = _log(rng, 1, 16)
        return dict(kind=kind, model=rng.choice(["llama-3.2-1b", "tinyllama"]), layers=4, batch=batch,
                    budget=rng.choice([257, 513]), prompt=_log(rng, 300, 32000 // batch if batch > 10 else 3000))
    if kind == "select":
        batch = _log(rng, 1, 24)
        return dict(kind=kind, model=rng.choice(["llama-3.2-1b", "llama-3.1-8b"]), batch=batch, budget=rng.choice([129, 257, 513]),
                    context=WINDOW + PAGE * max(8, _log(rng, 1000, min(32000, 260000 // batch)) // PAGE))
    design = rng.choice(["furitar", "bufodra"])
    size = rng.choice(["1b", "1b", "8b"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "float32"]) if size == "1b" else "bf16"
    layers = 2 if design == "furitar" else 4
    most = 16000 if dtype == "bf16" and size == "1b" else 6000 if dtype == "bf16" else 2500
    if kind == "prompts":
        batch = _log(rng, 1, 8)
        return dict(kind=kind, model=design + "-" + size, layers=layers, batch=batch, prompt=_log(rng, 65, most // batch), dtype=dtype)
    if kind == "steps":
        batch = _log(rng, 1, 64)
        return dict(kind=kind, model=design + "-" + size, layers=layers, batch=batch, prompt=_log(rng, 65, max(130, 4 * most // batch)),
                    dtype=dtype)
    batch = rng.randrange(2, 9)
    return dict(kind=kind, model=design + "-" + size, layers=layers, batch=batch, shortest=rng.randrange(1, 120),
                longest=rng.randrange(130, most // batch), steps=rng.randrange(2, 9), dtype=dtype)


# ------------------------------------------------------------------------------------------------------------- models and inputs
def _llama(case):
    """The zoo's entry with fewer layers, as plain numbers."""
    from magicdec_amd.Engine.model_core import transformer_configs
    c = dict(transformer_configs[case["model"]], n_layer=case.get("layers", 1), vocab_size=VOCAB)
    c.setdefault("n_local_heads", c["n_head"])
    return c


def _design(case):
    from magicdec_amd.Engine.designs import design_configs
    c = dict(design_configs[case["model"]], vocab=VOCAB)
    return dict(c, layers=c["layers"][:case["layers"]])


class _Draw:
    """Tensors from a seed, in a fixed order."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
        return torch.empty(shape, dtype=dtype, device=DEV).normal_(mean, std, generator=self.g)

    def tokens(self, *shape):
        return torch.randint(4, VOCAB, shape, device=DEV, generator=self.g)

    def head(self, emb, noise=0.02, tie=0.02):
        other = torch.randperm(VOCAB, device=DEV, generator=self.g)
        return (self.normal(*emb.shape, std=noise, dtype=torch.float32) + tie * emb[other].float()).to(emb.dtype)


def _llama_weights(c, d):
    dim, inter = c["dim"], c["intermediate_size"]
    D = dim // c["n_head"]
    qkv = (c["n_head"] + 2 * c["n_local_heads"]) * D
    w = {"tok_embeddings.weight": d.normal(VOCAB, dim)}
    for i in range(c["n_layer"]):
        p = "layers.%d." % i
        w[p + "attention.wqkv.weight"] = d.normal(qkv, dim, std=0.02)
        if c.get("qkv_bias"):
            w[p + "attention.wqkv.bias"] = d.normal(qkv, std=0.1)
        w[p + "attention.wo.weight"] = d.normal(dim, dim, std=0.02)
        w[p + "feed_forward.w1.weight"] = d.normal(inter, dim, std=0.02)
        w[p + "feed_forward.w3.weight"] = d.normal(inter, dim, std=0.02)
        w[p + "feed_forward.w2.weight"] = d.normal(dim, inter, std=0.02)
        w[p + "attention_norm.weight"] = d.normal(dim, mean=1.0, std=0.1)
        w[p + "ffn_norm.weight"] = d.normal(dim, mean=1.0, std=0.1)
    w["norm.weight"] = d.normal(dim, mean=1.0, std=0.1)
    w["output.weight"] = d.head(w["tok_embeddings.weight"])
    return w


def _design_weights(c, d, dtype):
    """The tensors of the design's model.safetensors."""
    W = c["width"]

    def mat(*shape):
        return d.normal(*shape, std=0.02, dtype=dtype)

    def norm(n):
        return d.normal(n, mean=1.0, std=0.1, dtype=dtype)
    furitar = c["architecture"] == "Furitar"
    t = {"embed": d.normal(VOCAB, W, std=1.0 if furitar else 0.02, dtype=dtype)}
    if furitar:
        t["pos"] = d.normal(c["max_positions"], W, std=0.3, dtype=dtype)
    else:
        t["bigram"], t["embed.norm"] = mat(c["embedding"]["bigram"]["buckets"] + 1, W), norm(W)
    for i, L in enumerate(c["layers"]):
        p, m, ff = "l%d." % i, L["mixer"], L["mlp"]["ff"]
        t[p + "norm1"] = norm(W)
        if furitar:
            H, G = m["heads"], m["kv_heads"]
            t[p + "shift"] = d.normal(W, mean=0.25, std=0.1, dtype=dtype)
            t[p + "mix.q"], t[p + "mix.k"], t[p + "mix.v"] = mat(H * m["dim"], W), mat(G * m["dim"], W), mat(G * m["vdim"], W)
            t[p + "mix.o"] = mat(W, H * m["vdim"])
            t[p + "mix.r1"] = d.normal(H, mean=0.5, std=0.1, dtype=dtype)
            t[p + "mix.r2"] = d.normal(H, mean=0.25, std=0.02, dtype=dtype)
            t[p + "norm2"] = norm(W)
            t[p + "mlp.up"], t[p + "mlp.down"] = mat(ff, W), mat(W, ff)
            t[p + "mlp.act"] = d.normal(2, std=0.3, dtype=dtype)
        else:
            H = m["heads"]
            t[p + "mix.dq"], t[p + "mix.dq.norm"] = mat(m["q_rank"], W), norm(m["q_rank"])
            if m.get("kv_from") is None:
                t[p + "mix.dkv"], t[p + "mix.dkv.norm"] = mat(m["kv_rank"] + m["rot_dim"], W), norm(m["kv_rank"])
            if L["type"] == "latent_attention":
                t[p + "mix.g"] = mat(H, W)
            t[p + "mix.uq"] = mat(H * (m["dim"] + m["rot_dim"]), m["q_rank"])
            t[p + "mix.uk"], t[p + "mix.uv"] = mat(H * m["dim"], m["kv_rank"]), mat(H * m["vdim"], m["kv_rank"])
            t[p + "mix.o"] = mat(W, H * m["vdim"])
            t[p + "mlp.gate"], t[p + "mlp.up"], t[p + "mlp.down"] = mat(ff, W), mat(ff, W), mat(W, ff)
    t["final.norm"] = norm(W)
    if furitar:
        t["head"] = d.head(t["embed"])
    return t


def _pages(tokens):
    return -(-tokens // PAGE)


def _context_rows(case, c, d):
    """Cache rows of a context: [pages, 2, KH, PAGE, D], the pages of a request side by side."""
    pages = case["batch"] * _pages(case["context"] + case["rows"])
    x = d.normal(pages, 2, c["n_local_heads"], PAGE, c["dim"] // c["n_head"], std=1.2)
    return x if case["kv"] == "bf16" else x.div_(FP8_SCALE).clamp_(-448, 448).to(torch.float8_e4m3fn)


def _draft_rows(case, c, d):
    """Rows of the compressed draft cache: [pages, 2, PAGE, KH, D]."""
    pages = case["batch"] * (case["budget"] // PAGE + 1)
    return d.normal(pages, 2, PAGE, c["n_local_heads"], c["dim"] // c["n_head"], std=1.2)


def _lengths(case):
    """Prompt lengths of a ragged batch: spread evenly over the range."""
    n = case["batch"] - 1
    return [case["shortest"] + (case["longest"] - case["shortest"]) * i // n for i in range(n + 1)]


def _dtype(case):
    return torch.float32 if case.get("dtype") == "float32" else torch.bfloat16


def _llama_engine(cls, case, c, weights, **kw):
    from magicdec_amd.Engine.model_core import transformer_configs
    name = "%s-%d-layers" % (case["model"], case["layers"])
    transformer_configs[name] = c
    engine = cls(dtype=torch.bfloat16, device=DEV, **kw)
    engine.load_model("no-checkpoint/%s/model.pth" % name, use_tp=False)
    engine.model.load_state_dict(weights, assign=True)
    return engine


def prepare(case, seed):
    d, kind = _Draw(seed), case["kind"]
    if kind in ("prompts", "steps", "ragged"):
        return _prepare_design(case, d)
    c = _llama(case)
    H, KH, D = c["n_head"], c["n_local_heads"], c["dim"] // c["n_head"]
    B = case["batch"]
    if kind == "select":
        from magicdec_amd import ops
        ppr, dpr = _pages(case["context"]), case["budget"] // PAGE + 1

        def table(n):
            return torch.arange(B * n, dtype=torch.int32, device=DEV), torch.arange(B + 1, dtype=torch.int32, device=DEV) * n
        return dict(kind=kind, q=d.normal(B * WINDOW, H, D, std=0.9), cache=d.normal(B * ppr, 2, KH, PAGE, D, std=0.9), table=table(ppr),
                    context=case["context"], budget=case["budget"], draft=torch.zeros(B * dpr, 2, PAGE, KH, D, dtype=torch.bfloat16, device=DEV),
                    draft_table=table(dpr), last=torch.ones(B, dtype=torch.int32, device=DEV), workspace=ops.AttnWorkspace(DEV))
    weights = _llama_weights(c, d)
    if kind == "decode":
        from magicdec_amd.Engine.SnapKV.backend import LMBackend
        rows, context = case["rows"], case["context"]
        engine = _llama_engine(LMBackend, case, c, weights, dec_len=rows)
        engine.compile()
        pages = _pages(context + rows)
        engine.setup_caches(max_batch_size=B, max_seq_length=pages * PAGE, kv_dtype=case["kv"], kv_layout="HND")
        for layer in engine.model.layers:
            kv = layer.attention.kv_cache
            kv.kv_cache.copy_(_context_rows(case, c, d))
            if case["kv"] == "fp8":
                kv.k_scale.fill_(FP8_SCALE)
                kv.v_scale.fill_(FP8_SCALE)
                kv.calibrated = True
        engine._t.map_pages(pages, context - (pages - 1) * PAGE)
        engine.cachelens.fill_(context)
        ids = d.tokens(B, rows)
        engine.inference(ids, benchmark=True)            # (the step's graph is captured at its first call)
        return dict(kind=kind, engine=engine, ids=ids)
    if kind == "draft":
        from magicdec_amd.Engine.SnapKV.backend_draft import LMBackend_Draft
        engine = _llama_engine(LMBackend_Draft, case, c, weights, draft_budget=case["budget"])
        engine.compile()
        engine.setup_caches(max_batch_size=B, max_seq_length=_pages(case["context"] + 64) * PAGE, draft_budget=case["budget"],
                            window_size=WINDOW)
        for layer in engine.model.layers:
            layer.attention.kv_cache.draft_cache.copy_(_draft_rows(case, c, d))
        engine.cachelens.fill_(case["context"])
        state = dict(kind=kind, engine=engine, ids=d.tokens(B, case["rows"]), rows=case["rows"])
        run(state)
        return state
    ids = d.tokens(B, case["prompt"])
    if kind == "encode":
        from magicdec_amd.Engine.SnapKV.backend import LMBackend
        engine = _llama_engine(LMBackend, case, c, weights, dec_len=1)
        engine.setup_caches(max_batch_size=B, max_seq_length=_pages(case["prompt"] + 80) * PAGE, kv_layout="HND")
    else:
        from magicdec_amd.Engine.StreamingLLM.backend_draft import LMBackend_Draft
        engine = _llama_engine(LMBackend_Draft, case, c, weights)
        engine.setup_caches(max_batch_size=B, draft_budget=case["budget"])
    return dict(kind=kind, engine=engine, ids=ids)


def _prepare_design(case, d):
    from magicdec_amd.Engine.SnapKV.backend import LMBackend
    from magicdec_amd.Engine.designs import design_configs
    c, dtype, B = _design(case), _dtype(case), case["batch"]
    name = "%s-%d-layers" % (case["model"], case["layers"])
    design_configs[name] = c
    engine = LMBackend(dtype=dtype, device=DEV)
    engine.load_model("no-checkpoint/%s/model.pth" % name, use_tp=False)
    model = engine.model
    model.output.weight = torch.nn.Parameter(model.output.weight.detach(), requires_grad=False)      # a tied head: not while loading
    model.load_state_dict(model.state_from_tensors(_design_weights(c, d, dtype)))
    model.tie_weights()
    if case["kind"] == "ragged":
        lengths = _lengths(case)
        engine.setup_caches(max_batch_size=B, max_seq_length=_pages(max(lengths) + case["steps"]) * PAGE,
                            num_pages=sum(_pages(n + case["steps"]) for n in lengths))
        return dict(kind="ragged", engine=engine, steps=case["steps"], sequences=[d.tokens(n + case["steps"]).cpu() for n in lengths])
    S = case["prompt"]
    ids = d.tokens(B, S)
    if case["kind"] == "steps":
        engine.compile()
    engine.setup_caches(max_batch_size=B, max_seq_length=_pages(S + 1) * PAGE)
    if case["kind"] == "prompts":
        return dict(kind="prompts", engine=engine, ids=ids)
    engine.encode(ids)
    step = d.tokens(B, 1)
    engine.inference(step, benchmark=True)
    return dict(kind="decode", engine=engine, ids=step)


# ------------------------------------------------------------------------------------------------------------- one pass
def run(s):
    if s["kind"] == "select":
        from magicdec_amd import ops
        places = ops.snapkv_select(s["q"], s["cache"], *s["table"], s["context"], WINDOW, s["budget"], 5, s["draft"], *s["draft_table"],
                                   s["last"], s["workspace"], kv_layout="HND")
        return {"places": places, "draft": s["draft"]}
    engine = s["engine"]
    if s["kind"] == "decode":
        tokens = engine.inference(s["ids"], benchmark=True)
    elif s["kind"] == "draft":
        tokens = engine.inference(s["ids"])
        engine.cachelens -= s["rows"]                    # rolled back, as after rejected tokens
        engine.draft_paged_kv_last_page_len -= s["rows"]
    elif s["kind"] == "ragged":
        return _run_ragged(s)
    else:
        tokens = engine.encode(s["ids"])
    return {"tokens": tokens, "logits": engine.model._last_logits}


def _run_ragged(s):
    engine, got = s["engine"], []
    for k in range(-1, s["steps"]):                      # the prompts, then one recorded token per sequence and step
        part = [(i, t[:t.numel() - s["steps"]] if k < 0 else t[t.numel() - s["steps"] + k:][:1]) for i, t in enumerate(s["sequences"])]
        got.append(engine.step(part, want=[[t.numel() - 1] for _, t in part]))
    for i in range(len(s["sequences"])):
        engine.end(i)
    return {"tokens": torch.stack([t for t, _ in got]), "logits": torch.stack([x for _, x in got])}


# ------------------------------------------------------------------------------------------------------------- bounds
def work(case):
    kind, B = case["kind"], case["batch"]
    if kind in ("prompts", "steps", "ragged"):
        return _work_design(case)
    c = _llama(case)
    H, KH, dim = c["n_head"], c["n_local_heads"], c["dim"]
    D = dim // H
    if kind == "select":
        S, keep = case["context"], case["budget"]
        return {"bytes": B * KH * D * 2 * (S + 4 * keep) + B * WINDOW * H * D * 2, "flops": 2.0 * B * WINDOW * H * S * D}
    layer = (H + 2 * KH) * D * dim + dim * dim + 3 * dim * c["intermediate_size"]
    L, head = c["n_layer"], VOCAB * dim
    if kind in ("decode", "draft"):
        M = B * case["rows"]
        T = case["context"] if kind == "decode" else case["budget"]
        each = 1 if case.get("kv") == "fp8" else 2
        return {"bytes": 2 * (L * layer + head) + L * B * T * KH * D * 2 * each + 2 * M * (dim + VOCAB),
                "flops": 2.0 * M * (L * layer + head) + 4.0 * L * M * H * D * T}
    S = case["prompt"]
    M, last = B * S, B * ((S - 1) % CHUNK + 1)
    seen = S / 2 if kind == "encode" else min(case["budget"], S / 2)
    kept = S if kind == "encode" else min(S, case["budget"])
    return {"bytes": 2 * (L * layer + head) + L * B * kept * KH * D * 4 + 2 * M * dim + 2 * last * VOCAB,
            "flops": 2.0 * M * L * layer + 2.0 * last * head + 4.0 * L * M * H * D * seen}


def _work_design(case):
    c, B = _design(case), case["batch"]
    W, size = c["width"], 4 if case["dtype"] == "float32" else 2
    furitar = c["architecture"] == "Furitar"
    params = row = pair = 0
    for L in c["layers"]:
        m, ff = L["mixer"], L["mlp"]["ff"]
        if furitar:
            params += W * (m["heads"] + m["kv_heads"]) * (m["dim"] + m["vdim"]) + 2 * W * ff
            row += m["kv_heads"] * (m["dim"] + m["vdim"])
            pair += m["heads"] * (m["dim"] + m["vdim"])
        else:
            own, gate = m.get("kv_from") is None, L["type"] == "latent_attention"
            params += W * (m["q_rank"] + own * (m["kv_rank"] + m["rot_dim"]) + gate * m["heads"])
            params += m["heads"] * (m["q_rank"] * (m["dim"] + m["rot_dim"]) + m["kv_rank"] * (m["dim"] + m["vdim"]) + m["vdim"] * W) + 3 * W * ff
            row += m["kv_rank"] + m["rot_dim"]
            pair += m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
    head = W * VOCAB
    if case["kind"] == "steps":
        M, heads, pairs, rows = B, B, B * case["prompt"], B * case["prompt"]
    elif case["kind"] == "prompts":
        M, heads, pairs, rows = B * case["prompt"], B, B * case["prompt"] ** 2 / 2, B * case["prompt"]
    else:
        total = [n + case["steps"] for n in _lengths(case)]
        M, heads, pairs, rows = sum(total), B * (case["steps"] + 1), sum(n * n / 2 for n in total), sum(total)
    return {"bytes": size * (params + head + row * rows + M * W + heads * VOCAB), "flops": 2.0 * M * params + 2.0 * heads * head + 2.0 * pairs * pair}


def tolerance(case):
    """16-bit rows between the launches of a few layers: 0.4 to 0.8 % off 64 bits, whatever the order of the sums.  32-bit throughout: 1e-6.
    The selection reproduces its reference's roundings bit by bit."""
    if case["kind"] == "select":
        return "exact"
    if case.get("dtype") == "float32":
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.0}
    return {"rel": 0.02, "max": 0.2, "differ": 0.01}


# ------------------------------------------------------------------------------------------------------------- 64 bits
def _rms(x, eps, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w.double()


def _mul(x, w):
    return x @ w.double().t()


def _turn(x, angle, amp=1.0):
    """Neighbouring pairs of x [T, ..., 2 p] turned by angle [T, p]."""
    angle = angle.view(angle.shape[0], *[1] * (x.dim() - 2), angle.shape[1])
    co, si = angle.cos() * amp, angle.sin() * amp
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * co - v * si, v * co + u * si], -1).flatten(-2)


def _rope(c, x, pos):
    """x [n, heads, D] at positions pos [n]."""
    D = c["dim"] // c["n_head"]
    f = c.get("rope_base", 10000) ** (-2.0 * torch.arange(D // 2, dtype=torch.float64, device=DEV) / D)
    scale = c.get("scaling_factor", 1.0)
    if c.get("high_freq_factor") is not None:
        lo, hi = c["low_freq_factor"], c["high_freq_factor"]
        keep = ((c["original_max_position_embeddings"] * f / (2 * math.pi) - lo) / (hi - lo)).clamp(0, 1)
        f = (1 - keep) * f / scale + keep * f
    else:
        f = f / scale
    return _turn(x, pos.double().view(-1, 1) * f)


def _attend(q, k, v, scale, first=None):
    """q [n, H, D]; k, v [T, KH, D]: query i sees the keys up to T - n + i (and from first[i] on)."""
    n, H, D = q.shape
    T, KH = k.shape[:2]
    out = torch.empty(n, H, v.shape[2], dtype=torch.float64, device=DEV)
    seen = torch.arange(T, device=DEV).view(1, -1) <= torch.arange(T - n, T, device=DEV).view(-1, 1)
    g = H // KH
    for h in range(KH):
        s = (q[:, h * g:(h + 1) * g].transpose(0, 1).reshape(g * n, D) @ k[:, h].t()).view(g, n, T) * scale
        p = torch.softmax(s.masked_fill_(~seen, float("-inf")), -1)
        out[:, h * g:(h + 1) * g] = (p.view(g * n, T) @ v[:, h]).view(g, n, -1).transpose(0, 1)
    return out


def _llama_exact(c, w, x, attend):
    """Layers over x [rows, dim]; attend(layer, q, k, v) -> [rows, H, D]."""
    H, KH, eps = c["n_head"], c["n_local_heads"], c.get("norm_eps", 1e-5)
    D = c["dim"] // H
    for i in range(c["n_layer"]):
        p = "layers.%d." % i
        z = _mul(_rms(x, eps, w[p + "attention_norm.weight"]), w[p + "attention.wqkv.weight"])
        if c.get("qkv_bias"):
            z = z + w[p + "attention.wqkv.bias"].double()
        q, k, v = z[:, :H * D].unflatten(1, (H, D)), z[:, H * D:(H + KH) * D].unflatten(1, (KH, D)), z[:, (H + KH) * D:].unflatten(1, (KH, D))
        x = x + _mul(attend(i, q, k, v).flatten(1), w[p + "attention.wo.weight"])
        y = _rms(x, eps, w[p + "ffn_norm.weight"])
        x = x + _mul(torch.nn.functional.silu(_mul(y, w[p + "feed_forward.w1.weight"])) * _mul(y, w[p + "feed_forward.w3.weight"]),
                     w[p + "feed_forward.w2.weight"])
    return x


def _answer(logits, shape):
    return {"tokens": logits.argmax(-1).view(shape), "logits": logits}


def exact(case, seed):
    d, kind, B = _Draw(seed), case["kind"], case["batch"]
    if kind == "select":
        return None                                      # its outputs are copies of input rows, in the order of 16-bit scores
    if kind in ("prompts", "steps", "ragged"):
        return _exact_design(case, d)
    c = _llama(case)
    w = _llama_weights(c, d)
    D, eps = c["dim"] // c["n_head"], c.get("norm_eps", 1e-5)

    def head(x):
        return _mul(_rms(x, eps, w["norm.weight"]), w["output.weight"])
    if kind in ("decode", "draft"):
        n, ctx = case["rows"], case["context"]
        store = [(_context_rows if kind == "decode" else _draft_rows)(case, c, d) for _ in range(c["n_layer"])]
        if kind == "decode":
            held = [(x.view(B, -1, 2, *x.shape[2:]).permute(2, 0, 1, 4, 3, 5), ctx) for x in store]     # [2, B, pages, PAGE, KH, D]
        else:
            held = [(x.view(B, -1, 2, *x.shape[2:]).transpose(0, 2).transpose(1, 2), case["budget"]) for x in store]
        unit = FP8_SCALE if case.get("kv") == "fp8" else 1.0
        ids = d.tokens(B, n)
        pos = torch.arange(ctx, ctx + n, device=DEV)

        def attend(i, q, k, v):
            out, (rows, T) = [], held[i]
            for b in range(B):
                at = slice(b * n, (b + 1) * n)
                old = [rows[j, b].flatten(0, 1)[:T].to(torch.float64) * unit for j in (0, 1)]
                out.append(_attend(_rope(c, q[at], pos), torch.cat([old[0], _rope(c, k[at], pos)]), torch.cat([old[1], v[at]]), D ** -0.5))
            return torch.cat(out)
        x = _llama_exact(c, w, w["tok_embeddings.weight"][ids.flatten()].double(), attend)
        return _answer(head(x), (B, n))
    S = case["prompt"]
    ids = d.tokens(B, S)
    tail = (S - 1) % CHUNK + 1
    x = w["tok_embeddings.weight"][ids].double()
    if kind == "encode":
        pos = torch.arange(S, device=DEV)

        def attend(i, q, k, v):
            q, k, v = (t.unflatten(0, (B, S)) for t in (q, k, v))
            return torch.cat([_attend(_rope(c, q[b], pos), _rope(c, k[b], pos), v[b], D ** -0.5) for b in range(B)])
        x = _llama_exact(c, w, x.flatten(0, 1), attend).unflatten(0, (B, S))[:, -tail:]
        return _answer(head(x.flatten(0, 1)), (B, tail))
    # StreamingLLM: portions of CHUNK tokens over `budget` cache slots; keys are rotated by their slot
    budget, KH = case["budget"], c["n_local_heads"]
    slots = [torch.zeros(2, B, budget, KH, D, dtype=torch.float64, device=DEV) for _ in range(c["n_layer"])]
    held = 0
    for at in range(0, S, CHUNK):
        part = x[:, at:at + CHUNK]
        n = part.shape[1]
        full = held + n > budget
        T = budget if full else held + n

        def attend(i, q, k, v):
            q, k, v = (t.unflatten(0, (B, n)) for t in (q, k, v))
            for j, new in ((0, k), (1, v)):
                if full:
                    slots[i][j][:, SINK:] = torch.cat([slots[i][j][:, SINK:], new], 1)[:, n:]
                else:
                    slots[i][j][:, held:T] = new
            pos = torch.arange(T, device=DEV)
            return torch.cat([_attend(_rope(c, q[b], pos[T - n:]), _rope(c, slots[i][0, b, :T], pos), slots[i][1, b, :T], D ** -0.5)
                              for b in range(B)])
        y = _llama_exact(c, w, part.flatten(0, 1), attend)
        held = T
    return _answer(head(y), (B, tail))


def _exact_design(case, d):
    c, dtype = _design(case), _dtype(case)
    t = _design_weights(c, d, dtype)
    forward = _furitar_exact if c["architecture"] == "Furitar" else _bufodra_exact
    if case["kind"] == "ragged":
        k = case["steps"]
        x = torch.stack([forward(c, t, d.tokens(n + k), k + 1) for n in _lengths(case)], 1)       # [steps + 1, B, vocab]
        return {"tokens": x.argmax(-1), "logits": x}
    ids = d.tokens(case["batch"], case["prompt"])
    if case["kind"] == "steps":
        ids = torch.cat([ids, d.tokens(case["batch"], 1)], 1)
    x = torch.cat([forward(c, t, row, 1) for row in ids])
    return _answer(x, (case["batch"], 1))


def _furitar_exact(c, t, tokens, last):
    eps, T = c["norm"]["eps"], tokens.numel()
    x = t["embed"][tokens].double() * c["embedding"]["scale"] + t["pos"][:T].double()
    i, j = torch.arange(T, device=DEV).view(-1, 1), torch.arange(T, device=DEV).view(1, -1)
    for n, L in enumerate(c["layers"]):
        p, m = "l%d." % n, L["mixer"]
        H, G, size = m["heads"], m["kv_heads"], m["mask"]["size"]
        h = _rms(x, eps, t[p + "norm1"])
        y = h + (torch.cat([torch.zeros_like(h[:1]), h[:-1]]) - h) * t[p + "shift"].double()
        q, k = (_rms(_mul(y, t[p + "mix." + s]).view(T, heads, -1), eps) for s, heads in (("q", H), ("k", G)))
        v = _mul(y, t[p + "mix.v"]).view(T, G, -1)
        unseen = (j > i) | (i // size != j // size)
        o = torch.empty(T, H, m["vdim"], dtype=torch.float64, device=DEV)
        for a in range(H):
            s = (q[:, a] @ k[:, a * G // H].t()) * m["scale"]
            s -= t[p + "mix.r1"][a].double() * torch.log1p(t[p + "mix.r2"][a].double() * (i - j).clamp(min=0))
            s.masked_fill_(unseen, float("-inf"))
            top = s.amax(-1, keepdim=True).clamp(min=0)
            e = torch.exp(s - top)
            o[:, a] = (e / (torch.exp(-top) + e.sum(-1, keepdim=True))) @ v[:, a * G // H]
        x = x + _mul(o.flatten(1), t[p + "mix.o"])
        z = _mul(_rms(x, eps, t[p + "norm2"]), t[p + "mlp.up"])
        right, left = torch.nn.functional.softplus(t[p + "mlp.act"].double())
        low = z.clamp(max=0)
        z = z / 2 + torch.where(z > 0, right * z * z, (0.5 + left) * (torch.expm1(low) - low))
        x = x + _mul(z, t[p + "mlp.down"])
    return _mul(_rms(x[-last:], eps, t["final.norm"]), t["head"]) * c["logit_scale"]


def _rotation(rot, T):
    """(angles [T, dims / 2], amplitude)"""
    n, base = rot["dims"], rot["base"]
    i = torch.arange(n // 2, dtype=torch.float64, device=DEV)
    f, amp, s = base ** (-2.0 * i / n), 1.0, rot.get("scaling")
    if s:
        lo, hi = (n * math.log(s["original"] / (2 * math.pi * s[k])) / (2 * math.log(base)) for k in ("fast", "slow"))
        lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), n - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        f, amp = f / s["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(s["factor"]) + 1.0
    return torch.arange(T, dtype=torch.float64, device=DEV).view(-1, 1) * f, amp


def _bufodra_exact(c, t, tokens, last):
    eps, T, big = c["norm"]["eps"], tokens.numel(), c["embedding"]["bigram"]
    pair = torch.cat([torch.full_like(tokens[:1], big["buckets"]),
                      (tokens[:-1] * big["mul_prev"] + tokens[1:] * big["mul_cur"]) % big["buckets"]])
    x = _rms(t["embed"][tokens].double() + t["bigram"][pair].double(), eps, t["embed.norm"])
    kept = {}
    for n, L in enumerate(c["layers"]):
        p, m = "l%d." % n, L["mixer"]
        H, D, R = m["heads"], m["dim"], m["kv_rank"]
        angle, amp = _rotation(m["rot"], T)
        h = _rms(x, eps, t[p + "norm1"])
        q = _mul(_rms(_mul(h, t[p + "mix.dq"]), eps, t[p + "mix.dq.norm"]), t[p + "mix.uq"]).view(T, H, -1)
        q = torch.cat([q[..., :D], _turn(q[..., D:], angle, amp)], -1)
        if m.get("kv_from") is None:
            z = _mul(h, t[p + "mix.dkv"])
            kept[n] = _rms(z[:, :R], eps, t[p + "mix.dkv.norm"]), _turn(z[:, R:], angle, amp)
        latent, r = kept[n if m.get("kv_from") is None else m["kv_from"]]
        k = torch.cat([_mul(latent, t[p + "mix.uk"]).view(T, H, D), r.unsqueeze(1).expand(T, H, -1)], -1)
        v = _mul(latent, t[p + "mix.uv"]).view(T, H, -1)
        o = _attend(q, k, v, m["scale"])
        if L["type"] == "latent_attention":
            o = o * torch.sigmoid(_mul(h, t[p + "mix.g"])).unsqueeze(-1)
        y = torch.nn.functional.gelu(_mul(h, t[p + "mlp.gate"]), approximate="tanh") * _mul(h, t[p + "mlp.up"])
        x = x + _mul(o.flatten(1), t[p + "mix.o"]) + _mul(y, t[p + "mlp.down"])
    cap = c["logit_softcap"]
    return cap * torch.tanh(_mul(_rms(x[-last:], eps, t["final.norm"]), t["embed"]) / cap)
