"""Balls with hundreds or thousands of edges to small ones, alone or side by
side (the edge between two has long rows at both ends), first or last in the
order of the ids, against the oracle, and recorded against that."""
import numpy as np
import pytest

import oracle
import pac

pytestmark = pytest.mark.gpu


def hub(leaves, seed, at=0.0):
    r = np.random.default_rng(seed)
    v = r.normal(size=(leaves, 3))
    big = 9.0 * np.sqrt(leaves / 300.0)
    b = np.empty((leaves + 1, 4), np.float32)
    b[0] = (at, 0, 0, big)
    b[1:, :3] = np.round((big + 0.8) * v / np.linalg.norm(v, axis=1)[:, None], 3)
    b[1:, 0] += np.float32(at)
    b[1:, 3] = 0.9
    return b


def balls(kind):
    if kind.startswith("hub"):
        return hub(int(kind[3:]), 5)
    if kind == "last":
        return hub(900, 6)[::-1].copy()
    two = np.concatenate([hub(700, 7), hub(800, 8, 22.0)])
    return two if kind == "two" else two[np.random.default_rng(9).permutation(len(two))]


@pytest.mark.parametrize("kind", ["hub191", "hub260", "hub1200", "hub3000",
                                  "last", "two", "shuffled"])
def test_lists(kind):
    print("case:", kind, flush=True)
    b = balls(kind)
    want, ost, _ = oracle.run(b, 0.4, 0.0)
    got = pac.compute(b, 0.4, 0.0)
    st = got.stats()
    assert (st.tri_candidates, st.tri_alpha) == (ost["T_cand"], ost["T_alpha"])
    assert (st.tet_candidates, st.tet_alpha) == (ost["K_cand"], ost["K_alpha"])
    g = pac.Graph(b, np.array([0, len(b)], np.int64), 0.4, 0.0)
    g.launch()
    for lists in (got.lists(), g.result().lists(0),
                  pac.compute(b, 0.4, 0.0, filtration=True).lists(),
                  pac.compute(b, 0.4, 0.0, chunk_balls=512).lists()):
        for d in (1, 2, 3):
            assert np.array_equal(lists[d], want[d]), d
