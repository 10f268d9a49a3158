import sys
r = lambda f: [l.split(" ", 1) for l in open("gpurun_out/" + f) if l[0].isdigit()]
a, b, c, d = r("rn1.txt"), r("rn2.txt"), r("ro1.txt"), r("ro2.txt")
import math
g = []
for w, x, y, z in zip(a, b, c, d):
    n, o = min(float(w[0]), float(x[0])), min(float(y[0]), float(z[0]))
    g.append(o / n)
    print("%9.1f -> %9.1f  %.3f  (new %s %s old %s %s) %s" % (o, n, o / n, w[0], x[0], y[0], z[0], w[1].strip()[:150]))
print("geomean %.4f" % math.exp(sum(map(math.log, g)) / len(g)))
