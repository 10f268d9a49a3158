import sys, os, torch
sys.path.insert(0, os.getcwd())
from magicdec_amd import ops
dev = "cuda:0"
def bench(B, KH, H, D, S, n, ragged):
    page = 128
    lens = [max(1, S * (i + 1) // B) for i in range(B)] if ragged else [S] * B
    pages = [-(-(l + n) // page) for l in lens]
    ptr = [0]
    for p in pages: ptr.append(ptr[-1] + p)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    spec = ops.XattnSpec(H, KH, D, D, D ** -0.5, 1e-5, chunk=0, sink=True, qk_norm=True)
    L = 4
    kc = [torch.empty(ptr[-1], KH, page, D, device=dev).normal_() for _ in range(L)]
    vc = [torch.empty(ptr[-1], KH, page, D, device=dev).normal_() for _ in range(L)]
    qkv = torch.empty(B * n, (H + 2 * KH) * D, device=dev).normal_()
    ws = ops.AttnWorkspace(dev)
    rows = ops.StepRows(i32([k * n for k in range(B + 1)]), i32(lens), n)
    idx, ip = i32(list(range(ptr[-1]))), i32(ptr)
    f = lambda i: ops.extended_attention(qkv, spec, kc[i % L], vc[i % L], rows, idx, ip, max(pages), ws)
    for i in range(4): o = f(i)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for i in range(20): o = f(i)
    ts = []
    for _ in range(7):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record(); g.replay(); b.record(); b.synchronize(); ts.append(a.elapsed_time(b) / 20 * 1e3)
    return sorted(ts)[3]
import random
rng = random.Random(int(sys.argv[1]))
import math
for k in range(60):
    KH, H, D = rng.choice([(8, 32, 64), (8, 32, 64), (4, 16, 128), (8, 32, 128), (2, 8, 256), (8, 8, 256), (4, 16, 96)])
    B = int(round(math.exp(rng.uniform(0, math.log(40))))); S = int(round(math.exp(rng.uniform(math.log(20), math.log(3000))))); n = rng.choice([1, 1, 1, 2, 4])
    if B * S > 60000: S = 60000 // B
    c = (B, KH, H, D, S, n, rng.choice([0, 1]))
    if len(sys.argv) > 2:
        KH, H, D = rng.choice([(8, 8, 256), (8, 24, 256), (4, 16, 192)]); B = rng.randrange(1, 12) * 8 // KH; c = (B, KH, H, D, rng.randrange(100, 2500), n, rng.choice([0, 1]))
    print(*c, "us: %.2f" % bench(*c), flush=True)
