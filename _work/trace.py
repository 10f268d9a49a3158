# per-kernel gaps of the last pass from rocprofv3's kernel trace CSV
import csv, sys
rows = list(csv.DictReader(open(sys.argv[1])))
rows.sort(key=lambda r: int(r["Start_Timestamp"]))
n = int(sys.argv[2])   # launches to show from the end
rows = rows[-n:]
prev = None
for r in rows:
    s, e = int(r["Start_Timestamp"]), int(r["End_Timestamp"])
    print("%8.2f gap %6.2f  %-70s g%sx%sx%s/%s vgpr %s lds %s" % ((e - s) / 1e3, (s - prev) / 1e3 if prev else 0, r["Kernel_Name"][:70], r["Grid_Size_X"], r["Grid_Size_Y"], r["Grid_Size_Z"], r["Workgroup_Size_X"], r.get("VGPR_Count"), r.get("LDS_Block_Size")))
    prev = e
