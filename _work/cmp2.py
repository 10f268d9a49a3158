import torch, sys
a, b = torch.load(sys.argv[1]), torch.load(sys.argv[2])
bad = 0
for i, (x, y) in enumerate(zip(a, b)):
    for u, v in zip(x, y):
        if u.dtype == torch.bfloat16: u, v = u.view(torch.int16), v.view(torch.int16)
        if not torch.equal(u, v): bad += 1; print("differs", i, (u != v).sum().item())
print("compared", len(a), len(b), "bad", bad)
sys.exit(bad > 0)
