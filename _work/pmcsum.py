import csv, sys
from collections import defaultdict
d = defaultdict(dict)
for r in csv.DictReader(open(sys.argv[1])):
    d[(int(r["Dispatch_Id"]), r["Kernel_Name"][:60])][r["Counter_Name"]] = float(r["Counter_Value"])
last = {}
for (i, k), v in sorted(d.items()): last[k] = v
for k, v in last.items():
    if "snapkv" in k: print(k, {a: "%.3g" % b for a, b in v.items()})
