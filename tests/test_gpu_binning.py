"""The order (cell, id) from counted cells and from sorted keys: grids on
either side of the rule between them, one full cell, shuffled ids, single
balls and repeated positions, against the oracle."""
import numpy as np
import pytest

import oracle
import pac

pytestmark = pytest.mark.gpu


def same(b, solvent=1.4):
    got = pac.compute(b, solvent, 0.0)
    want, _, _ = oracle.run(b, solvent, 0.0)
    lists = got.lists()
    for d in (1, 2, 3):
        assert np.array_equal(lists[d], want[d]), d
    return got.stats().grid_cells


@pytest.mark.parametrize("n,far,counted", [
    (400, 0.0, True), (400, 120.0, True), (400, 260.0, False),
    (400, 700.0, False), (3000, 0.0, True), (3000, 120.0, False),
    (3000, 260.0, False), (3000, 700.0, False)])
def test_grids(n, far, counted):
    print("case:", n, far, flush=True)
    b = pac.synth_globule(n, seed=n)
    b[n // 2:, :3] += np.float32(far)
    b = b[np.random.default_rng(n).permutation(n)]
    cells = same(b)
    assert (cells <= 4 * n + 65536) == counted


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 257, 600])
def test_one_cell(n):
    """small balls in the cells of a large one"""
    r = np.random.default_rng(n)
    b = np.empty((n, 4), np.float32)
    b[:, :3] = np.round(r.uniform(0, 2.5, (n, 3)), 2)
    b[:, 3] = 0.15
    b[n // 2] = b[0]
    b[n // 3] = (9, 9, 9, 5)
    same(b, 0.0)


@pytest.mark.parametrize("sizes", [(1, 300, 2, 1500), (700, 1, 1, 900)])
def test_batch_cells(sizes):
    parts = [pac.synth_globule(k, seed=k) for k in sizes]
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    got = pac.compute_batch(np.concatenate(parts), off, 1.4, 0.0)
    for q, p in enumerate(parts):
        want, _, _ = oracle.run(p, 1.4, 0.0)
        for d in (1, 2, 3):
            assert np.array_equal(got.lists(q)[d], want[d]), (q, d)
