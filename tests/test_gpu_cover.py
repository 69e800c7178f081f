"""Emptiness decisions spared by covered edges (tet candidates counted but
not listed, triangles and edges failing without a scan) against the oracle,
row for row: balls swallowed by larger ones, alpha below and above zero,
alpha-edge counts around one enumeration block (256), alpha triangles on
either side of the count from which they are listed before their scans
(131072, between 1300 and 1500 balls), and the same input as a batch, in
chunks, recorded and in FP64."""
import numpy as np
import pytest

import oracle
import pac

pytestmark = pytest.mark.gpu


def _balls(n, seed, spread):
    b = pac.synth_globule(n, None, 1.1, seed=seed)
    r = np.random.default_rng(seed)
    big = r.random(n) < 0.1
    b[big, 3] = (b[big, 3] * np.float32(spread)).astype(np.float32)
    return b


def _same(got, want, what):
    for d in (1, 2, 3):
        assert np.array_equal(got[d], want[d]), "%s: dim %d" % (what, d)


@pytest.mark.parametrize("n,spread,s,a", [
    (3, 1.0, 1.4, 0.0), (24, 1.6, 1.4, 0.0), (40, 1.0, 0.4, 0.0),
    (257, 2.2, 1.4, 0.0), (900, 1.8, 1.0, -1.5), (900, 1.5, 0.0, 4.0),
    (1300, 1.0, 1.4, 0.0), (1500, 1.0, 1.4, 0.0), (2500, 2.0, 1.4, 0.0)])
def test_covered_edges(n, spread, s, a):
    print("case:", n, spread, s, a, flush=True)
    b = _balls(n, 40 + n, spread)
    want, st, _ = oracle.run(b, s, a)
    for prec in (pac.PREC_STAGED, pac.PREC_PLAIN_FP64):
        res = pac.compute(b, s, a, precision=prec)
        _same(res.lists(), want, "prec %d" % prec)
        got = res.stats()
        assert got.tet_candidates == st["K_cand"]
        assert got.tet_alpha == st["K_alpha"]
    _same(pac.compute_f64(b.astype(np.float64), s, a).lists(),
          oracle.run(b.astype(np.float64), s, a)[0], "fp64")
    _same(pac.compute(b, s, a, chunk_balls=512).lists(), want, "chunked")
    off = np.array([0, n, n, 2 * n])
    two = np.concatenate([b, b])
    g = pac.Graph(two, off, s, a)
    for rep in range(3):
        g.launch()
        rec = g.result()
        bat = pac.compute_batch(two, off, s, a)
        for m in (0, 2):
            _same(rec.lists(m), want, "recorded %d" % rep)
            _same(bat.lists(m), want, "batch")
        assert rec.stats().tet_alpha == bat.stats().tet_alpha == 2 * st["K_alpha"]
