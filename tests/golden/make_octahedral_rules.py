"""Prints the table kRules of spheresimulator_amd/csrc/shtables.cpp: quadrature
rules on the sphere with octahedral symmetry (the structure is Lebedev's, Zh.
Vychisl. Mat. Mat. Fiz. 16 (1976)), one per order of a far-field level.

The polynomials on the sphere that the group of the octahedron leaves alone are
spanned by (x^4 + y^4 + z^4)^a (x y z)^2b, so a rule of degree L that is a sum of
orbits has to give their means for 4a + 6b <= L.  Unknown are the weights of the
orbits and the places of those that are free.  Least squares from random starts
finds a root with positive weights, Newton's method in 40 digits sharpens it.

Run from anywhere: python3 tests/golden/make_octahedral_rules.py  (about 2 minutes; needs mpmath)
"""
import itertools

import mpmath as mp
import numpy as np
from scipy.optimize import least_squares

mp.mp.dps = 40
# order of the level: degree of its rule, then how many orbits of (0,0,1), (0,1,1), (1,1,1),
# (t,t,u), (0,t,u) and (t,u,v).  Order 6 takes order 7's (that of degree 13 has a negative weight).
RULES = {1: (3, 1, 0, 0, 0, 0, 0), 2: (5, 1, 0, 1, 0, 0, 0), 3: (7, 1, 1, 1, 0, 0, 0), 4: (9, 1, 0, 1, 0, 1, 0),
         5: (11, 1, 1, 1, 1, 0, 0), 7: (15, 1, 0, 1, 2, 1, 0), 8: (17, 1, 0, 1, 3, 1, 0), 9: (19, 1, 1, 1, 3, 0, 1),
         10: (21, 1, 1, 1, 3, 1, 1)}


def mean(a, b):
    """Mean of (x^4 + y^4 + z^4)^a (x y z)^2b over the sphere."""
    total = mp.mpf(0)
    for i in range(a + 1):
        for j in range(a - i + 1):
            e = [4 * i + 2 * b, 4 * j + 2 * b, 4 * (a - i - j) + 2 * b]
            m = mp.factorial(a) / (mp.factorial(i) * mp.factorial(j) * mp.factorial(a - i - j))
            total += m * mp.fprod(mp.fac2(k - 1) for k in e) / mp.fac2(sum(e) + 1)
    return total


def points(orbits, free):
    """One point of each orbit and the number of its images; free: their coordinates t (and u)."""
    a1, a2, a3, b, c, d = orbits
    f = iter(free)
    out = [(6, (0, 0, 1))] * a1 + [(12, (0, mp.sqrt(2) / 2, mp.sqrt(2) / 2))] * a2
    out += [(8, (1 / mp.sqrt(3),) * 3)] * a3
    for _ in range(b):
        t = next(f)
        out.append((24, (t, t, mp.sqrt(1 - 2 * t * t))))
    for _ in range(c):
        t = next(f)
        out.append((24, (0, t, mp.sqrt(1 - t * t))))
    for _ in range(d):
        t, u = next(f), next(f)
        out.append((48, (t, u, mp.sqrt(1 - t * t - u * u))))
    return out


def start(orbits, moments, rng):
    """Least squares in double precision from random places."""
    nw, nf = sum(orbits), orbits[3] + orbits[4] + 2 * orbits[5]
    fixed = [(6, (0, 0, 1.0))] * orbits[0] + [(12, (0, 0.5 ** 0.5, 0.5 ** 0.5))] * orbits[1]
    fixed += [(8, (3 ** -0.5,) * 3)] * orbits[2]

    def pts(g):
        g, out = list(g), list(fixed)
        for _ in range(orbits[3]):
            t = g.pop(0)
            out.append((24, (np.sin(t) / 2 ** 0.5, np.sin(t) / 2 ** 0.5, np.cos(t))))
        for _ in range(orbits[4]):
            t = g.pop(0)
            out.append((24, (0.0, np.sin(t), np.cos(t))))
        for _ in range(orbits[5]):
            t, u = g.pop(0), g.pop(0)
            out.append((48, (np.sin(t) * np.cos(u), np.sin(t) * np.sin(u), np.cos(t))))
        return out

    def res(v):
        ps = pts(v[nw:])
        s4, s6 = [sum(c ** 4 for c in p) for _, p in ps], [27.0 * np.prod(p) ** 2 for _, p in ps]
        return [sum(w * m * x ** a * y ** b for w, (m, _), x, y in zip(v, ps, s4, s6)) - float(t) * 27.0 ** b
                for (a, b), t in moments]

    while True:
        v0 = np.concatenate([rng.uniform(0.7, 1.3, nw) / sum(m for m, _ in pts(np.ones(nf))),
                             rng.uniform(0, np.pi / 2, nf)])
        r = least_squares(res, v0, xtol=1e-15, ftol=1e-15, gtol=1e-15, max_nfev=300)
        if max(abs(r.fun)) > 1e-13 or min(r.x[:nw]) <= 0:
            continue
        ps = [tuple(np.abs(p)) for _, p in pts(r.x[nw:])]
        images = set()  # a genuine rule: no orbit has fallen onto another or onto one with fewer images
        for p in ps:
            images |= {tuple(round(s * c, 9) + 0.0 for s, c in zip(sg, q)) for q in itertools.permutations(p)
                       for sg in itertools.product((1, -1), repeat=3)}
        if len(images) == sum(m for m, _ in pts(r.x[nw:])):
            free = []
            for p, n in zip(ps[sum(orbits[:3]):], [1] * orbits[3] + [2] * orbits[4] + [3] * orbits[5]):
                free += {1: [p[0]], 2: [p[1]], 3: [p[0], p[1]]}[n]
            return [float(x) for x in r.x[:nw]] + free


def main():
    rng = np.random.default_rng(0)
    for q, (degree, *orbits) in RULES.items():
        moments = [((a, b), mean(a, b)) for b in range(degree // 6 + 1) for a in range((degree - 6 * b) // 4 + 1)]
        nw = sum(orbits)

        def res(*v):
            ps = points(orbits, v[nw:])
            return [sum(w * m * sum(c ** 4 for c in p) ** a * mp.fprod(p) ** (2 * b) for w, (m, p) in zip(v, ps)) - t
                    for (a, b), t in moments]

        v = list(mp.findroot(res, start(orbits, moments, rng), tol=1e-35, maxsteps=30))
        ps = points(orbits, v[nw:])
        print("    // order %d: %d points (degree %d)" % (q, sum(m for m, _ in ps), degree))
        rows = ["{%s}" % ", ".join(repr(float(x)) for x in sorted(p) + [w]) for w, (_, p) in zip(v, ps)]
        print("    {" + ",\n     ".join(rows) + "},", flush=True)


if __name__ == "__main__":
    main()
