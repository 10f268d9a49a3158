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
for c in [(1, 8, 32, 64, 130, 1, 0), (1, 8, 32, 64, 600, 1, 0), (1, 8, 32, 64, 2000, 1, 0), (2, 8, 32, 64, 1000, 1, 0), (4, 8, 32, 64, 500, 1, 0), (6, 8, 32, 64, 1508, 1, 1), (6, 8, 32, 64, 1500, 1, 0), (6, 8, 32, 64, 300, 1, 0), (8, 8, 32, 64, 700, 1, 1), (12, 8, 32, 64, 600, 1, 0), (16, 8, 32, 64, 2000, 1, 0), (32, 8, 32, 64, 600, 1, 0), (4, 8, 32, 128, 1000, 1, 0), (2, 4, 16, 128, 2000, 4, 0), (4, 2, 8, 256, 900, 1, 0), (6, 8, 32, 64, 1500, 4, 0)]:
    print(*c, "us: %.2f" % bench(*c), flush=True)
