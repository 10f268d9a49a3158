import sys, os, torch
sys.path.insert(0, os.getcwd())
from perf import cases
for c in cases.listed():
    s = cases.prepare(c, 1)
    for _ in range(2): cases.run(s)
    torch.cuda.synchronize()
    torch.empty(3, device="cuda:0").uniform_().erfinv_()
    for _ in range(4): cases.run(s)
    torch.cuda.synchronize()
    torch.empty(3, device="cuda:0").uniform_().erfinv_()
    torch.cuda.synchronize()
    del s; torch.cuda.empty_cache()
    print("done", c["name"], flush=True)
