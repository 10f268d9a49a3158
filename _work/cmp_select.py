# outputs of the select of two trees over drawn sizes and value ranges, bit by bit: python cmp_select.py out.pt  (run in a tree's root)
import sys, os, random, torch
sys.path.insert(0, os.getcwd())
from magicdec_amd import ops
dev = "cuda:0"
rng = random.Random(7)
out = []
for n in range(40):
    D = rng.choice([64, 128]); g = rng.choice([1, 2, 3, 4, 5, 7, 8]); W = rng.choice([16, 32]) if g > 1 else 16
    if g == 1: W = 8
    if (g * W) % 16 or 8 * g < W or g * W > 256: W = 16 if 8 * g >= 16 else 8
    if (g * W) % 16: continue
    KH = rng.choice([1, 2, 8]); B = rng.choice([1, 2, 5, 9]); S = rng.choice([160, 700, 1531, 4128, 9000])
    budget = rng.choice([65, 129, 257]); page = 128; std = rng.choice([0.05, 0.5, 0.9, 1.5, 3.0, 8.0, 20.0])
    pool = rng.choice([1, 5, 5, 7, 131])
    if budget - W > S - W or budget >= S: budget = 65
    fp8 = rng.random() < 0.3
    H = KH * g; ppr = -(-S // page); dpr = budget // page + 1
    gen = torch.Generator(device=dev).manual_seed(n)
    q = torch.empty(B * W, H, D, device=dev).normal_(0, std, generator=gen).bfloat16()
    kv = torch.empty(B * ppr, 2, KH, page, D, device=dev).normal_(0, 0.9, generator=gen).bfloat16()
    kw = {}
    draft = torch.zeros(B * dpr, 2, page, KH, D, dtype=torch.bfloat16, device=dev)
    ar = lambda k: torch.arange(k, dtype=torch.int32, device=dev)
    print(n, B, KH, g, D, W, S, budget, pool, std, flush=True)
    idx, sc = ops.snapkv_select(q, kv, ar(B * ppr), ar(B + 1) * ppr, S, W, budget, pool, draft, ar(B * dpr), ar(B + 1) * dpr,
                                torch.full((B,), budget - (dpr - 1) * page, dtype=torch.int32, device=dev), ops.AttnWorkspace(dev), return_scores=True, kv_layout="HND")
    out.append((idx.cpu(), sc.cpu(), draft.cpu()))
torch.cuda.synchronize()
torch.save(out, sys.argv[1])
