"""Tets of balls that are all in one another's rows, on either side of the
rows' length (63) where the per-edge masks give way to merges, and of such a
cluster inside an ordinary globule, against the oracle."""
import numpy as np
import pytest

import oracle
import pac

pytestmark = pytest.mark.gpu


def same(b, solvent, **kw):
    got = pac.compute(b, solvent, 0.0, **kw)
    want, ost, _ = oracle.run(b, solvent, 0.0)
    lists = got.lists()
    for d in (1, 2, 3):
        assert np.array_equal(lists[d], want[d]), d
    st = got.stats()
    if not kw:
        assert st.tet_candidates == ost["K_cand"]
        assert st.tet_alpha == ost["K_alpha"]


def cluster(n, seed, box=8.0):
    r = np.random.default_rng(seed)
    b = np.empty((n, 4), np.float32)
    b[:, :3] = np.round(r.uniform(0, box, (n, 3)), 3)
    b[:, 3] = np.round(r.uniform(1.0, 1.9, n), 2)
    return b


@pytest.mark.parametrize("n", [5, 33, 34, 63, 64, 65, 66, 72])
@pytest.mark.parametrize("solvent", [6.0, 20.0])
def test_cluster(n, solvent):
    print("case:", n, solvent, flush=True)
    same(cluster(n, n), solvent)


@pytest.mark.parametrize("kw", [{}, {"chunk_balls": 256}])
def test_cluster_in_globule(kw):
    b = np.concatenate([pac.synth_globule(700, seed=3), cluster(66, 9, 4.0)])
    same(b, 1.4, **kw)
