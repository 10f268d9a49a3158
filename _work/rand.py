# time of given cases (dicts) in a tree: python rand.py file.json (run in the tree's root); us per pass, median of 5 x n
import sys, os, json, time, torch
sys.path.insert(0, os.getcwd())
sys.path.insert(0, os.path.join(os.getcwd(), "perf"))
from perf import cases
for c in json.load(open(sys.argv[1])):
    s = cases.prepare(c, 1)
    for _ in range(3): cases.run(s)
    torch.cuda.synchronize()
    t = time.perf_counter(); cases.run(s); torch.cuda.synchronize(); one = time.perf_counter() - t
    n = max(3, min(200, int(0.1 / one)))
    ts = []
    for _ in range(5):
        t = time.perf_counter()
        for _ in range(n): cases.run(s)
        torch.cuda.synchronize()
        ts.append((time.perf_counter() - t) / n * 1e6)
    ts.sort()
    print("%.1f %s" % (ts[2], json.dumps(c)), flush=True)
    del s; torch.cuda.empty_cache()
