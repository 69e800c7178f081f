"""Adjoint where balls lie in no simplex, in a few, and in hundreds or
thousands (a large ball among many small ones), against the FP64 reference
gradient; two calls give the same bits."""
import numpy as np
import pytest

import pac
import adjoint_ref as ref

pytestmark = pytest.mark.gpu


def hub(leaves, seed):
    r = np.random.default_rng(seed)
    v = r.normal(size=(leaves, 3))
    b = np.empty((leaves + 2, 4), np.float32)
    b[0] = (0, 0, 0, 9.0)
    b[1:-1, :3] = np.round(9.6 * v / np.linalg.norm(v, axis=1)[:, None], 3)
    b[1:-1, 3] = 1.1
    b[-1] = (40, 40, 40, 1.0)
    return b


@pytest.mark.parametrize("leaves", [30, 500, 4000])
def test_hub(leaves):
    print("case:", leaves, flush=True)
    b = hub(leaves, leaves)
    res = pac.compute(b, 0.4, 0.0)
    L = res.lists()
    lists = {2: L[2].astype(np.int64), 3: L[3].astype(np.int64)}
    pos, r = ref.balls_f64(b, 0.4)
    T, K = len(lists[2]), len(lists[3])
    assert T > 0 and K > 0
    rng = np.random.default_rng(1)
    g = {2: rng.uniform(-1, 1, T), 3: rng.uniform(-1, 1, K)}
    dxyz, dr = res.adjoint(g[2], g[3])
    rp, rr = ref.gradient(pos, r, lists, g)
    # (1e-9 of the largest entry, as the other adjoint tests)
    scale = max(np.abs(rp).max(), np.abs(rr).max())
    assert np.abs(dxyz - rp).max() <= 1e-9 * scale
    assert np.abs(dr - rr).max() <= 1e-9 * scale
    assert not dxyz[-1].any() and dr[-1] == 0
    again = res.adjoint(g[2], g[3])
    assert np.array_equal(again[0], dxyz) and np.array_equal(again[1], dr)
