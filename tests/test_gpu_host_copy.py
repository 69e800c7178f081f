"""Lists copied to host memory: sizes around a 16 KiB segment and around half
the ring of segments (2 MiB), rows that start at any word, several threads at
once and pinned destinations, against copies that stay on the device."""
import threading

import numpy as np
import pytest
import torch

import pac

pytestmark = pytest.mark.gpu


def on_device(r, dim):
    m = r.counts()[dim]
    t = torch.empty((m, dim + 1), dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    r.copy_list_to(dim, t.data_ptr())
    return t.cpu().numpy()


@pytest.mark.parametrize("n", [2, 7, 262, 1500, 3001, 12000, 40001])
def test_lists_and_values(n):
    print("case:", n, flush=True)
    r = pac.compute(pac.synth_globule(n, seed=n), 1.4, 0.0, filtration=True)
    host = r.lists()
    for d in (1, 2, 3):
        m = r.counts()[d]
        assert np.array_equal(host[d], on_device(r, d))
        pinned = torch.full((m + 1, d + 1), -7, dtype=torch.int32).pin_memory()
        r.copy_list_to(d, pinned.data_ptr())
        assert np.array_equal(pinned[:m].numpy(), host[d])
        assert (pinned[m:] == -7).all()
        rho = torch.empty(m, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        r.copy_alpha_to(d, rho.data_ptr())
        assert np.array_equal(r.alpha_values(d), rho.cpu().numpy())


def test_batch_rows_in_local_ids():
    sizes = [3, 1, 5000, 2, 801, 4003, 17, 2500]
    parts = [pac.synth_globule(k, seed=11 + k) for k in sizes]
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    b = pac.compute_batch(np.concatenate(parts), off, 1.4, 0.0)
    for q, p in enumerate(parts):
        got, want = b.lists(q), pac.compute(p, 1.4, 0.0).lists()
        for d in (1, 2, 3):
            assert np.array_equal(got[d], want[d]), (q, d)


def test_threads():
    rs = [pac.compute(pac.synth_globule(k, seed=k), 1.4, 0.0)
          for k in (500, 6000, 15000)]
    want = [[on_device(r, d) for d in (1, 2, 3)] for r in rs]
    bad = []

    def work(r, w):
        for _ in range(5):
            got = r.lists()
            bad.extend(d for d in (1, 2, 3)
                       if not np.array_equal(got[d], w[d - 1]))

    ts = [threading.Thread(target=work, args=a) for a in zip(rs, want)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
    pac.memory_trim()
    assert np.array_equal(rs[0].lists()[1], want[0][0])
