import csv, sys, re
from collections import defaultdict
sys.path.insert(0, "/root/repo")
names = [m for m in re.findall(r'dict\(name="([^"]+)"', open("/root/repo/perf/cases.py").read())]
rows = list(csv.DictReader(open(sys.argv[1])))
rows.sort(key=lambda r: int(r["Start_Timestamp"]))
marks = [i for i, r in enumerate(rows) if "erfinv" in r["Kernel_Name"]]
assert len(marks) == 2 * len(names), (len(marks), len(names))
print("""Kernel times of perf/cases.py's listed cases: rocprofv3 --kernel-trace --stats, four passes each after two warm ones, microseconds per
pass, launches per pass, microseconds per launch, kernel and grid / workgroup.  "span" includes the gaps between launches, which the
profiler widens ("now" of the design notes' table is measured without it).
""")
for k, name in enumerate(names):
    sub = rows[marks[2 * k] + 1:marks[2 * k + 1]]
    sub = [r for r in sub if "uniform" not in r["Kernel_Name"] and not ("distribution" in r["Kernel_Name"] and int(r["Grid_Size_X"]) <= 256)]
    t = lambda r: int(r["End_Timestamp"]) - int(r["Start_Timestamp"])
    span = (int(sub[-1]["End_Timestamp"]) - int(sub[0]["Start_Timestamp"])) / 4e3
    busy = sum(map(t, sub)) / 4e3
    print("=== %s: span %.1f us, busy %.1f us, %d kernels/pass" % (name, span, busy, round(len(sub) / 4)))
    d = defaultdict(lambda: [0, 0])
    for r in sub:
        kn = r["Kernel_Name"].replace("(anonymous namespace)::", "")
        kn = "library " + re.search(r"MT\d+x\d+x\d+", kn).group(0) if kn.startswith("Cijk") else kn.split("(")[0] if not kn.startswith("_Z") else kn
        key = "%s g%sx%sx%s/%s" % (kn[:70], r["Grid_Size_X"], r["Grid_Size_Y"], r["Grid_Size_Z"], r["Workgroup_Size_X"])
        d[key][0] += 1; d[key][1] += t(r)
    for key, v in sorted(d.items(), key=lambda x: -x[1][1])[:18]:
        print("  %9.1f us %7.1f x %8.2f  %s" % (v[1] / 4e3, v[0] / 4, v[1] / v[0] / 1e3, key))
