"""Candidates whose orthosphere power equals alpha exactly (a cubic lattice of
equal balls), decided by the last stage of the filters and kept, against the
oracle: eagerly, and through a recorded batch."""
import numpy as np
import pytest

import oracle
import pac

pytestmark = pytest.mark.gpu


def lattice(k):
    g = np.arange(k) * 2.0
    xyz = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    return np.c_[xyz, np.ones(len(xyz))].astype(np.float32)


@pytest.mark.parametrize("alpha", [0.0, 1.0, 2.0])  # edges, triangles, tets
@pytest.mark.parametrize("k", [2, 6])
@pytest.mark.parametrize("prec", [pac.PREC_STAGED, pac.PREC_PLAIN_FP64])
def test_ties(k, alpha, prec):
    print("case:", k, alpha, prec, flush=True)
    b = lattice(k)
    got = pac.compute(b, 0.0, alpha, precision=prec)
    want, ost, _ = oracle.run(b, 0.0, alpha)
    assert ost["exact_filter"] > 0
    for d in (1, 2, 3):
        assert np.array_equal(got.lists()[d], want[d]), d
    st = got.stats()
    assert (st.edge_alpha, st.tri_alpha, st.tet_alpha) == (
        ost["E_alpha"], ost["T_alpha"], ost["K_alpha"])


@pytest.mark.parametrize("alpha", [1.0, 2.0])
def test_ties_recorded(alpha):
    b = lattice(4)
    off = np.array([0, len(b)], np.int64)
    g = pac.Graph(b, off, 0.0, alpha)
    g.launch()
    got = g.result().lists(0)
    want, _, _ = oracle.run(b, 0.0, alpha)
    for d in (1, 2, 3):
        assert np.array_equal(got[d], want[d]), d
