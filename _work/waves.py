import sys, os, time, torch
sys.path.insert(0, os.getcwd())
from magicdec_amd import ops, _lib
dev = "cuda:0"
lib = _lib.load()
def bench(B, KH, H, D, S, n, nw, fp8=False):
    lib.md_debug_set_attn_waves(nw)
    page = 128; ppr = -(-(S + n) // page)
    L = 4
    caches = [torch.empty(B * ppr, 2, KH, page, D, device=dev, dtype=torch.bfloat16).normal_() for _ in range(L)]
    q = torch.empty(B * n, H, D, device=dev, dtype=torch.bfloat16).normal_()
    ar = lambda k: torch.arange(k, dtype=torch.int32, device=dev)
    qo, idx, ptr = ar(B + 1) * n, ar(B * ppr), ar(B + 1) * ppr
    last = torch.full((B,), (S + n - 1) % page + 1, dtype=torch.int32, device=dev)
    ws = ops.AttnWorkspace(dev)
    f = lambda i: ops.paged_attention(q, caches[i % L], qo, idx, ptr, last, n, ppr, ws, causal=True, kv_layout="HND")
    for i in range(4): o = f(i)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for i in range(40): o = f(i)
    ts = []
    for _ in range(7):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record(); g.replay(); b.record(); b.synchronize(); ts.append(a.elapsed_time(b) / 40 * 1e3)
    return sorted(ts)[3]
for B, KH, H, D, S, n in [(64, 8, 32, 64, 257, 1), (32, 8, 32, 64, 257, 1), (16, 8, 32, 64, 257, 1), (64, 8, 32, 64, 513, 1), (64, 8, 32, 64, 129, 1), (64, 4, 32, 64, 257, 1), (8, 8, 32, 64, 513, 1), (1, 12, 12, 64, 129, 1), (1, 12, 12, 64, 1000, 1), (16, 8, 32, 128, 500, 4), (64, 8, 32, 128, 300, 4)]:
    print(B, KH, H, D, S, n, " 4: %.2f  8: %.2f" % (bench(B, KH, H, D, S, n, 4), bench(B, KH, H, D, S, n, 8)), flush=True)
