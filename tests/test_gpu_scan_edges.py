"""Ball counts on either side of a scan tile (2048) and of the scans that run
in one launch (16 tiles, 32768 balls), lists against the oracle."""
import numpy as np
import pytest

import oracle
import pac

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2047, 2048, 2049, 4097, 32768, 32769])
def test_scan_tile_edges(n):
    print("case:", n, flush=True)
    b = pac.synth_globule(n, seed=n)
    got = pac.compute(b, 0.0, 1.0).lists()
    want, _, _ = oracle.run(b, 0.0, 1.0)
    for d in (1, 2, 3):
        assert np.array_equal(got[d], want[d]), d
