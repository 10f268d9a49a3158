import sys, os, torch
sys.path.insert(0, os.getcwd())
from magicdec_amd import ops
dev = "cuda:0"; out = []
for n, (B, KH, g, D, W, S, budget) in enumerate([(64, 4, 4, 64, 32, 1000, 129), (40, 8, 4, 128, 32, 1056, 257), (33, 8, 8, 64, 16, 2064, 129), (5, 2, 5, 128, 32, 3000, 129), (70, 4, 2, 64, 16, 990, 65)]):
    H = KH * g; page = 128; ppr = -(-S // page); dpr = budget // page + 1
    gen = torch.Generator(device=dev).manual_seed(n)
    q = torch.empty(B * W, H, D, device=dev).normal_(0, 0.9, generator=gen).bfloat16()
    kv = torch.empty(B * ppr, 2, KH, page, D, device=dev).normal_(0, 100, generator=gen).clamp_(-448, 448).to(torch.float8_e4m3fn)
    sc = [torch.rand(KH, device=dev, generator=gen) * 0.01 + 0.004 for _ in range(2)]
    draft = torch.zeros(B * dpr, 2, page, KH, D, dtype=torch.bfloat16, device=dev)
    ar = lambda k: torch.arange(k, dtype=torch.int32, device=dev)
    print(n, flush=True)
    idx, s = ops.snapkv_select(q, kv, ar(B * ppr), ar(B + 1) * ppr, S, W, budget, 5, draft, ar(B * dpr), ar(B + 1) * dpr,
                               torch.full((B,), budget - (dpr - 1) * page, dtype=torch.int32, device=dev), ops.AttnWorkspace(dev), return_scores=True, kv_scales=tuple(sc), kv_layout="HND")
    out.append((idx.cpu(), s.cpu(), draft.cpu()))
torch.save(out, sys.argv[1])
