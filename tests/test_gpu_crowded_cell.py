"""Many small balls in the one cell of a grid that a large ball sets.  Cells of
thousands against the oracle; inputs refused for their edge candidates, and
inputs without edges, end without work that grows with the square of a cell
(a million balls would walk 10^12 ids before the refusal)."""
import time

import numpy as np
import pytest

import oracle
import pac

pytestmark = pytest.mark.gpu


def crowd(n, radius=0.15, big=50.0, dtype=np.float32):
    r = np.random.default_rng(n)
    b = np.empty((n, 4), dtype)
    b[:, :3] = np.round(r.uniform(0, 40, (n, 3)), 3)
    b[:, 3] = radius
    if big:
        b[n // 3] = (300, 300, 300, big)
    return b


@pytest.mark.parametrize("n", [7, 8, 9, 1023, 2049, 6000])
def test_order(n):
    print("case:", n, flush=True)
    b = crowd(n)
    want, _, _ = oracle.run(b, 0.3, 0.0)
    off = np.array([0, n, n + 9], np.int64)
    two = np.concatenate([b, crowd(9)])
    for got in (pac.compute(b, 0.3, 0.0).lists(),
                pac.compute_f64(b.astype(np.float64), 0.3, 0.0).lists()
                if n < 3000 else None,
                pac.compute_batch(two, off, 0.3, 0.0).lists(0)):
        for d in (1, 2, 3):
            if got is not None:
                assert np.array_equal(got[d], want[d]), d


@pytest.mark.parametrize("n,dtype", [(200000, np.float32),
                                     (1000000, np.float32),
                                     (300000, np.float64)])
def test_refused_at_once(n, dtype):
    print("case:", n, dtype.__name__, flush=True)
    pac.compute(crowd(100), 0.3, 0.0)
    b = crowd(n, dtype=dtype)
    run = pac.compute if dtype == np.float32 else pac.compute_f64
    t = time.perf_counter()
    with pytest.raises(pac.PacError) as e:
        run(b, 0.3, 0.0)
    assert e.value.code == pac.PAC_ERR_OVERFLOW
    assert time.perf_counter() - t < 1.0


def test_no_edges():
    """largest radius squared + alpha < 0: nothing is enumerated"""
    print("case: no edges", flush=True)
    n = 300000
    b = crowd(n, radius=50.0, big=0)
    pac.compute(b[:100], -49.0, -2.0)
    t = time.perf_counter()
    r = pac.compute(b, -49.0, -2.0)
    assert time.perf_counter() - t < 1.0
    assert [int(c) for c in r.counts()] == [n, 0, 0, 0]
