import sys, os, statistics, torch
sys.path.insert(0, os.getcwd())
from perf import cases
from magicdec_amd.Engine import model_core
def engine(case, limit):
    model_core.LAST_LEVEL_CACHE = limit
    s = cases.prepare(case, 1)
    model_core.LAST_LEVEL_CACHE = 256 << 20
    return s
def need(s):
    m = s["engine"].model
    return sum(p.data.numel() * p.data.element_size() for k, p in m._packed.items()) / 1e6
todo = [dict(kind="draft", model="llama-3.2-1b", layers=L, batch=64, budget=257, context=4000, rows=1) for L in (2, 3, 4, 5, 6, 8, 12, 16)]
todo += [dict(kind="draft", model="llama-3.2-1b", layers=L, batch=40, budget=257, context=4000, rows=1) for L in (3, 4, 16)]
todo += [dict(kind="decode", model="llama-3.1-8b", layers=L, batch=64, context=500, rows=1, kv="bf16") for L in (1, 2, 8)]
todo += [dict(kind="decode", model="Qwen2.5-7b", layers=L, batch=48, context=500, rows=1, kv="bf16") for L in (1, 4)]
todo += [dict(kind="decode", model="68m", layers=2, batch=64, context=500, rows=1, kv="bf16")]
for c in todo:
    c["name"] = "x"
    try:
        ss = {"off": engine(c, 1 << 60), "on": engine(c, 0)}
    except Exception as e:
        print("skip", c, repr(e)[:200], flush=True); continue
    t = {"off": [], "on": []}
    for r in range(12):
        for k, s in ss.items():
            for _ in range(5): cases.run(s)
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(40): cases.run(s)
            b.record(); b.synchronize()
            t[k].append(a.elapsed_time(b) * 25)
    m = {k: statistics.median(v) for k, v in t.items()}
    print("%s %s layers %d batch %d: %.0f MB  off %.1f (%.1f-%.1f) on %.1f (%.1f-%.1f)  %.3f" % (c["kind"], c["model"], c["layers"], c["batch"], need(ss["on"]),
          m["off"], min(t["off"]), max(t["off"]), m["on"], min(t["on"]), max(t["on"]), m["off"] / m["on"]), flush=True)
    del ss, s
    torch.cuda.empty_cache()
