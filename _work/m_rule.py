import sys, os, copy, statistics, torch
sys.path.insert(0, os.getcwd())
from magicdec_amd import ops
lib = ops._lib.load()
BF = torch.bfloat16
dev = "cuda:0"
torch.manual_seed(0)
def graphs(M, tiles, K, epi):
    N = tiles * 32
    n = max(2, min(64, (800 << 20) // (N * K * 2)))
    x = torch.randn(M, K, device=dev).to(BF)
    w = torch.randn(N, K, device=dev).mul_(0.05).to(BF)
    base = ops.PackedWeight(w, swiglu=epi == "swiglu")
    pws = []
    for _ in range(n):
        p = copy.copy(base); p.data = base.data.clone(); pws.append(p)
    resid = torch.randn(M, N, device=dev).to(BF)
    out = torch.empty(M, N // 2 if epi == "swiglu" else N, device=dev, dtype=BF)
    def go():
        for p in pws:
            if epi == "swiglu": ops.fused_linear(x, p, swiglu=True, out=out)
            elif epi == "resid": ops.fused_linear(x, p, resid=resid, out=out)
            else: ops.fused_linear(x, p, out=out)
    gs = {}
    for knob in (0, 11):
        lib.md_debug_set_fused_nw(knob)
        go(); torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g): go()
        gs[knob] = g
    lib.md_debug_set_fused_nw(0)
    t = {0: [], 11: []}
    for r in range(9):
        for k, g in gs.items():
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record(); g.replay(); b.record(); b.synchronize()
            if r > 1: t[k].append(a.elapsed_time(b) * 1e3 / n)
    return {k: statistics.median(v) for k, v in t.items()}, n, (pws, resid, out, x)
full = len(sys.argv) > 1
tl = [258, 264, 272, 288, 304, 320, 336, 352, 368, 384, 400, 416, 448, 480, 504, 512]
for K in (256, 1024, 2048, 4096):
    for epi in ("plain", "swiglu", "resid"):
        for M in (17, 32):
            line = []
            for tiles in tl:
                r, n, _ = graphs(M, tiles, K, epi)
                line.append("%d %.2f/%.2f %.3f" % (tiles, r[11], r[0], r[11] / r[0]))
                del _
            print("K %d %s M %d | " % (K, epi, M) + " | ".join(line), flush=True)
