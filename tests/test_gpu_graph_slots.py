"""A recorded batch accepts another input with the counts it was recorded for,
without headroom: a slab of balls and pairs of balls apart from it, moved by
whole cells from behind the slab to beside it.  Cells, rows and simplices stay
as they are, but the 64 edges that a wave of the triangle enumeration takes are
of other rows, whose bitmaps find 675 more false hits for 36,463 triangles."""
import numpy as np
import pytest

import pac

pytestmark = pytest.mark.gpu

N, PAIRS, X, Z = 20000, 1900, 60, 32  # cells of side 2 (largest radius 1)


def slab_and_pairs(beside):
    r = np.random.default_rng(3)
    slab = np.empty((N, 4), np.float32)
    slab[:, :3] = r.integers(0, 64, (N, 3)) / 64.0 * np.array([X, X, Z])
    slab[:, :3] = np.floor(slab[:, :3] * 64) / 64
    slab[:, 3] = 1.0
    k = np.arange(PAIRS)
    at = np.c_[X + 4.0 + 4.0 * (k // (X * Z // 4)), 2.0 * (k % (X // 2)),
               2.0 * (k // (X // 2) % (Z // 2)) + (0 if beside else Z + 8)]
    pairs = np.empty((2 * PAIRS, 4), np.float32)
    pairs[0::2, :3] = pairs[1::2, :3] = at
    pairs[1::2, 0] += 0.125
    pairs[:, 3] = 0.25
    ends = np.array([[0, 0, -8, 1], [X + 28, X, 2 * Z + 16, 1]], np.float32)
    return np.concatenate([ends[:1], slab, pairs, ends[1:]])


def test_moved_pairs_no_headroom():
    print("case: pairs behind and beside a slab", flush=True)
    behind, beside = slab_and_pairs(False), slab_and_pairs(True)
    off = np.array([0, len(behind)], np.int64)
    for first, second in ((behind, beside), (beside, behind)):
        g = pac.Graph(first, off, 0.0, 0.0, headroom=0.0)
        for b in (first, second, first):
            g.set_input(b)
            g.launch()
            r = g.result()
            want = pac.compute(b, 0.0, 0.0)
            for d in (1, 2, 3):
                assert np.array_equal(r.lists(0)[d], want.lists()[d]), d
            st, ref = r.stats(), want.stats()
            for f in ("edge_candidates", "edge_alpha", "tri_candidates",
                      "tri_alpha", "tet_candidates", "tet_alpha"):
                assert getattr(st, f) == getattr(ref, f), f
