"""A recorded batch's results taken on one thread while eager runs, with the
scratch they give back between their kernels, go on in another: both
threads' lists as when they run alone."""
import threading

import numpy as np
import pytest

import pac

pytestmark = pytest.mark.gpu


def test_results_beside_eager_runs():
    print("case: graph results beside eager runs", flush=True)
    sizes = (9000, 40, 14000)
    x = np.concatenate([pac.synth_globule(k, seed=k) for k in sizes])
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    b = pac.synth_globule(23000, seed=8)
    graph = pac.Graph(x, off, 1.4, 0.0, batch_balls=10000)
    want = [r.lists(m) for r in [pac.compute_batch(x, off, 1.4, 0.0)]
            for m in range(3)]
    alone = pac.compute(b, 1.4, 0.0).lists()
    bad = []

    def same(got, ref, what):
        bad.extend((what, d) for d in (1, 2, 3)
                   if not np.array_equal(got[d], ref[d]))

    def recorded():
        for rep in range(30):
            graph.launch()
            r = graph.result()
            for m in range(3):
                same(r.lists(m), want[m], ("recorded", rep, m))

    def eager():
        for rep in range(30):
            same(pac.compute(b, 1.4, 0.0).lists(), alone, ("eager", rep))

    ts = [threading.Thread(target=f) for f in (recorded, eager, eager)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
