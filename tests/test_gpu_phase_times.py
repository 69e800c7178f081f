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


def test_no_tets():
    """balls of one plane: the triangles' test is most of the run"""
    print("case: no tets", flush=True)
    b = pac.synth_globule(1500, seed=2)
    b[:, 2] = 0
    pac.compute(b, 1.4, 0.0)
    st = pac.compute(b, 1.4, 0.0).stats()
    t = phases(st)
    assert st.tri_alpha > 0 and st.tet_alpha == 0
    assert t["AC2 test for triangles"] > t["AC2 test for tetrahedra"]
    assert t["AC2 test for edges"] > 0


def test_no_triangles():
    """separate pairs: the edges' test has a time of its own"""
    print("case: no triangles", flush=True)
    b = np.zeros((40000, 4), np.float32)
    k = np.arange(20000)
    b[0::2, 0], b[0::2, 1], b[0::2, 2] = 8 * (k % 30), 8 * (k // 30 % 30), 8 * (k // 900)
    b[1::2] = b[0::2]
    b[1::2, 0] += 1
    b[:, 3] = 1.5
    pac.compute(b, 0.0, 0.0)
    st = pac.compute(b, 0.0, 0.0).stats()
    t = phases(st)
    assert st.edge_alpha == 20000 and st.tri_alpha == 0
    assert t["AC2 test for edges"] > 0 and t["Potential triangles"] > 0


def test_transfer():
    """pinned memory is copied behind the call: 32 MB take the bus at least
    0.2 ms (160 GB/s would), however soon the copy's call returns"""
    print("case: transfer", flush=True)
    import torch
    n = 2000000
    b = np.zeros((n, 4), np.float32)
    k = np.arange(n)
    b[:, 0], b[:, 1], b[:, 2] = 4 * (k % 128), 4 * (k // 128 % 128), 4 * (k // 16384)
    b[:, 3] = 1.0
    pinned = torch.from_numpy(b).pin_memory()
    for x in (b, pinned.numpy()):
        pac.compute(x, 0.0, 0.0)
        t = phases(pac.compute(x, 0.0, 0.0).stats())
        assert 0.2 < t["Data transfer"] < 50, t
    dev = pinned.cuda()
    torch.cuda.synchronize()
    r = pac.compute_device(dev.data_ptr(), n, 0.0, 0.0)
    assert phases(r.stats())["Data transfer"] == 0
