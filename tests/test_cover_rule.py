"""The rule that spares emptiness scans, in rationals: where a triangle of
alpha edges has value > alpha and a negative barycentric coordinate of its
orthocentre at vertex k, every alpha simplex with the edge opposite k has k's
power strictly below its value (so it is not empty), ties included.
"""
import itertools
import random
from fractions import Fraction as F

import pytest


def _sphere(balls):
    """(barycentric weights, centre, value) of the smallest orthosphere, or
    None when the centres are affinely dependent."""
    p0, w0 = balls[0]
    a = [[q - o for q, o in zip(p, p0)] for p, _ in balls[1:]]
    m = len(a)
    rows = [[sum(x * y for x, y in zip(a[i], a[j])) for j in range(m)]
            + [(sum(x * x for x in a[i]) + w0 - balls[i + 1][1]) / 2]
            for i in range(m)]
    for c in range(m):
        piv = next((r for r in range(c, m) if rows[r][c] != 0), None)
        if piv is None:
            return None
        rows[c], rows[piv] = rows[piv], rows[c]
        rows[c] = [x / rows[c][c] for x in rows[c]]
        for r in range(m):
            if r != c and rows[r][c]:
                rows[r] = [x - rows[r][c] * y for x, y in zip(rows[r], rows[c])]
    lam = [r[m] for r in rows]
    off = [sum(l * v[q] for l, v in zip(lam, a)) for q in range(3)]
    c = [o + q for o, q in zip(p0, off)]
    return [1 - sum(lam)] + lam, c, sum(x * x for x in off) - w0


@pytest.mark.parametrize("seed,grid,rmax", [(1, 3, 4), (2, 4, 6), (3, 6, 6),
                                            (4, 2, 3), (5, 5, 9)])
def test_covered_edge_has_no_empty_simplex(seed, grid, rmax):
    rng = random.Random(seed)
    covered = decided = 0
    for _ in range(60):
        pts = rng.sample(list(itertools.product(range(grid + 1), repeat=3)), 6)
        b = [(tuple(F(x) for x in p), F(rng.randint(1, rmax), 2) ** 2)
             for p in pts]
        alpha = F(rng.randint(-4, 8), 4)
        sph = {s: _sphere([b[v] for v in s])
               for m in (2, 3, 4) for s in itertools.combinations(range(6), m)}
        ok = {s: v is not None and v[2] <= alpha for s, v in sph.items()}
        for t in itertools.combinations(range(6), 3):
            if sph[t] is None or ok[t] or not all(
                    ok[e] for e in itertools.combinations(t, 2)):
                continue
            for q, k in enumerate(t):
                if sph[t][0][q] >= 0:
                    continue
                edge = set(t) - {k}
                covered += 1
                for s, v in sph.items():
                    if ok[s] and edge <= set(s):
                        power = sum((x - y) ** 2 for x, y in
                                    zip(b[k][0], v[1])) - b[k][1]
                        assert k not in s and power < v[2], (b, alpha, t, s)
                        decided += 1
    assert covered > 10 and decided > 20
