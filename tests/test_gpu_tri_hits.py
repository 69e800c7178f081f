"""Triangles of rows on either side of the lengths (64, 128) at which the hit
masks grow a word and give way to merges, of a segment of 64 edges whose last
row runs far past it, and of many balls of one edge each, against the
oracle."""
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
    assert st.tri_candidates == ost["T_cand"]
    assert st.tri_alpha == ost["T_alpha"]


def star(leaves, seed):
    """a ball with an edge to each of `leaves` others, which have few edges
    with one another"""
    r = np.random.default_rng(seed)
    v = r.normal(size=(leaves, 3))
    b = np.empty((leaves + 1, 4), np.float32)
    b[0] = (0, 0, 0, 9.0)
    b[1:, :3] = np.round(10.0 * v / np.linalg.norm(v, axis=1)[:, None], 3)
    b[1:, 3] = 0.8
    return b


@pytest.mark.parametrize("leaves", [3, 62, 63, 64, 65, 66, 127, 128, 129, 190,
                                    191, 192, 193, 260, 300, 390])
def test_star(leaves):
    print("case:", leaves, flush=True)
    same(star(leaves, leaves), 0.4)


@pytest.mark.parametrize("n", [33, 97, 130, 131, 160])
def test_dense(n):
    """rows of up to n - 1 ids, most pairs and triples alpha"""
    print("case:", n, flush=True)
    r = np.random.default_rng(n)
    b = np.empty((n, 4), np.float32)
    b[:, :3] = np.round(r.uniform(0, 9, (n, 3)), 3)
    b[:, 3] = 1.5
    same(b, 2.2)


def test_pairs_and_triples():
    """64 different first balls in a segment: isolated pairs and triples"""
    r = np.random.default_rng(5)
    parts = []
    for k in range(300):
        c = np.array([k % 7, (k // 7) % 7, k // 49]) * 12.0
        m = 2 + k % 2
        parts.append(np.c_[c + r.uniform(0, 1.5, (m, 3)), np.full(m, 1.5)])
    same(np.round(np.concatenate(parts), 3).astype(np.float32), 0.5)
