# time of the select over drawn sizes: python sel_rand.py (in a tree's root)
import sys, os, random, torch
sys.path.insert(0, os.getcwd())
from magicdec_amd import ops
dev = "cuda:0"; rng = random.Random(11)
W, page = 32, 128
def log(lo, hi):
    import math
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
for n in range(36):
    D, KH, g = rng.choice([(64, 8, 4), (128, 8, 4), (128, 4, 7), (64, 4, 8), (128, 8, 8), (64, 8, 5)])
    B = log(1, 32); S = W + page * max(8, log(1000, min(32000, 260000 // B)) // page); budget = 257
    H = KH * g; ppr = -(-S // page); dpr = budget // page + 1
    gen = torch.Generator(device=dev).manual_seed(n)
    q = torch.empty(B * W, H, D, device=dev).normal_(0, 0.9, generator=gen).bfloat16()
    kv = torch.empty(B * ppr, 2, KH, page, D, dtype=torch.bfloat16, device=dev).normal_(0, 0.9, generator=gen)
    ar = lambda k: torch.arange(k, dtype=torch.int32, device=dev)
    draft = torch.zeros(B * dpr, 2, page, KH, D, dtype=torch.bfloat16, device=dev)
    ws = ops.AttnWorkspace(dev); t1, t2, t3, t4 = ar(B * ppr), ar(B + 1) * ppr, ar(B * dpr), ar(B + 1) * dpr
    last = torch.ones(B, dtype=torch.int32, device=dev)
    f = lambda: ops.snapkv_select(q, kv, t1, t2, S, W, budget, 5, draft, t3, t4, last, ws, kv_layout="HND")
    for _ in range(3): f()
    ts = []
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(5): f()
        b.record(); b.synchronize(); ts.append(a.elapsed_time(b) * 200)
    print("B %d S %d D %d KH %d g %d" % (B, S, D, KH, g), "us %.1f" % sorted(ts)[2], flush=True)
