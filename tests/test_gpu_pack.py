"""Triangle and edge emptiness packed by blocks, on either side of the number
of simplices it starts from, with blocks that hold more undecided ones than
threads, against one phase over everything and (the smaller ones) the
oracle."""
import numpy as np
import pytest

import oracle
import pac

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,alpha", [(1200, 0.0), (2300, 0.0), (9000, 0.0),
                                     (12000, -1.2)])
@pytest.mark.parametrize("filt", [False, True])
def test_packed(n, alpha, filt):
    """(filtration tests every triangle and edge that is not covered)"""
    print("case:", n, alpha, filt, flush=True)
    b = pac.synth_globule(n, seed=n)
    got = pac.compute(b, 1.4, alpha, filtration=filt)
    one = pac.compute(b, 1.4, alpha, filtration=filt, ac2_budget=-1)
    for d in (1, 2, 3):
        assert np.array_equal(got.lists()[d], one.lists()[d]), d
    if filt:
        for x, y in zip(got.filtration(), one.filtration()):
            assert np.array_equal(x, y)
    if n < 3000:
        want, ost, _ = oracle.run(b, 1.4, alpha)
        for d in (1, 2, 3):
            assert np.array_equal(got.lists()[d], want[d]), d


@pytest.mark.parametrize("n", [260, 400])
def test_many_left(n):
    """a cluster: rows and columns of triangles no ball covers"""
    r = np.random.default_rng(n)
    v = r.normal(size=(n, 3))
    b = np.empty((n, 4), np.float32)
    b[:, :3] = np.round(6.0 * v / np.linalg.norm(v, axis=1)[:, None], 3)
    b[:, 3] = 1.0
    got = pac.compute(b, 2.0, 0.0)
    want, ost, _ = oracle.run(b, 2.0, 0.0)
    for d in (1, 2, 3):
        assert np.array_equal(got.lists()[d], want[d]), d
