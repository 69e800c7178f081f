"""Phase times of a run: each phase that did work has its time, and under its
own name."""
import numpy as np
import pytest

import pac

pytestmark = pytest.mark.gpu


def phases(st):
    return dict(zip(pac.PHASE_LABELS, st.phase_ms))


@pytest.mark.parametrize("batch_balls", [0, 5000])
def test_batch(batch_balls):
    print("case: batch", batch_balls, flush=True)
    sizes = (3000, 4000, 200)
    x = np.concatenate([pac.synth_globule(k, seed=k) for k in sizes])
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    t = phases(pac.compute_batch(x, off, 1.4, 0.0,
                                 batch_balls=batch_balls).stats())
    assert all(t[k] > 0 for k in pac.PHASE_LABELS[1:]), t
    assert sum(t.values()) < 100
