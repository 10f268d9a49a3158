import sys, os, torch
sys.path.insert(0, os.getcwd())
from perf import cases
names = sys.argv[1].split(",")
n = int(sys.argv[2])
for c in cases.listed():
    if c["name"] in names:
        s = cases.prepare(c, 1)
        for _ in range(3): cases.run(s)
        torch.cuda.synchronize()
        for _ in range(n): cases.run(s)
        torch.cuda.synchronize()
        print("done", c["name"], flush=True)
