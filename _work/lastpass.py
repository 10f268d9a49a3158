import csv, sys
from collections import defaultdict
rows = list(csv.DictReader(open(sys.argv[1])))
rows.sort(key=lambda r: int(r["Start_Timestamp"]))
# passes separated by marker kernel: argmax
idx = [i for i, r in enumerate(rows) if 'argmax' in r["Kernel_Name"]]
sub = rows[idx[-2] + 1: idx[-1] + 1]
print(len(sub), (int(sub[-1]["End_Timestamp"]) - int(sub[0]["Start_Timestamp"])) / 1e3, sum(int(r["End_Timestamp"]) - int(r["Start_Timestamp"]) for r in sub) / 1e3)
d = defaultdict(lambda: [0, 0])
for r in sub:
    k = (r["Kernel_Name"].replace("(anonymous namespace)::", "").replace("at::native::", "")[:70], r["Grid_Size_X"], r["Grid_Size_Y"])
    d[k][0] += 1; d[k][1] += int(r["End_Timestamp"]) - int(r["Start_Timestamp"])
for k, v in sorted(d.items(), key=lambda x: -x[1][1]): print("%8.1f %4d x %7.1f %s" % (v[1] / 1e3, v[0], v[1] / v[0] / 1e3, k))
