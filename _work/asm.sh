cd /root/repo/magicdec_amd/csrc && /opt/rocm/bin/hipcc -O3 -std=c++17 --offload-arch=gfx950 -Xclang -target-feature -Xclang -packed-fp32-ops -ffp-contract=off --cuda-device-only -S snapkv.hip -o /root/repo/_work/snap.s 2>/dev/null; cd /root/repo; python3 - <<'P'
import re
from collections import Counter
t=open('_work/snap.s').read()
f=t[t.index('_ZN12_GLOBAL__N_119snapkv_accum_kernelILi64ELb0ELi2ELi8ELi32EEEvNS_10SnapParamsE:'):]
f=f[:f.index('.Lfunc_end')]
open('_work/accum.s','w').write(f)
for b in re.split(r'\n(?=\.LBB)',f):
    n=len(re.findall(r'\n\s+[vsdgb]_?\w+',b))
    if 'mfma' in b or 'ds_read_b64' in b or 'permlane' in b:
        print(b[:12],n,dict(Counter(re.findall(r'\n\s+(\w+)',b)).most_common(30)))
P
