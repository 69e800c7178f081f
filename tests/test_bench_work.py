"""CPU: the work bench.py charges its kernels with is work a run does: alpha
tets that are counted but not scanned are charged no set-up, and every kernel
that can be the dominant one has its measured traffic."""
import json
import os
import sys
from types import SimpleNamespace

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


def test_setups_of_scanned_tets_only():
    st = SimpleNamespace(edge_candidates=5, tri_candidates=7, tet_candidates=11,
                         ac2_pairs=[1000, 300, 20], tet_alpha=19_000_000,
                         tets_final=600_000)
    units, setups = bench.work_units(st)
    assert units["tet_ac2"] == 1000 and units["edge_ac2"] == 20
    assert setups == 600_000
    su = bench.WORK_MODEL["flops"]["tet_ac2_setup"]["f32"]
    per = bench.WORK_MODEL["flops"]["tet_ac2"]["f32"]
    assert bench.kernel_flops("tet_ac2", 1000, setups, False) == (
        1000 * per + 600_000 * su, 0.0)
    assert bench.kernel_flops("tri_ac2", 300, setups, True) == (
        0.0, 300 * bench.WORK_MODEL["flops"]["tri_ac2"]["f32"])


def test_traffic_of_every_kernel():
    path = os.path.join(ROOT, "profiles", "hbm_traffic_globule100k.json")
    per_run = json.load(open(path))["bytes_per_run"]
    assert set(per_run) == set(bench.KERNEL_KEYS)
    assert all(v > 0 for v in per_run.values())
