"""CPU: device code that reads its Stage again from the kernel's arguments
stays in the bodies of kernels (anywhere else that address means nothing), also
where nothing is inlined by choice, and those kernels take the Stage first."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_kernel_bodies_only(tmp_path):
    ll = tmp_path / "k_ac2.ll"
    subprocess.run(
        [HIPCC, "--offload-arch=gfx950", "-O1", "-fno-inline", "-std=c++17",
         "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops", "-DPAC_BALL_F64=1", "--cuda-device-only",
         "-emit-llvm", "-S", "k_ac2.hip", "-o", str(ll)], check=True,
        cwd=os.path.join(ROOT, "parallelac-xmp_amd", "csrc"),
        capture_output=True)
    where, readers = "", []
    for line in ll.read_text().splitlines():
        if line.startswith("define"):
            where = line
        elif "call" in line and "@llvm.amdgcn.kernarg.segment.ptr()" in line:
            readers.append(where)
    assert len(readers) > 10
    for f in readers:
        assert " amdgpu_kernel " in f, f[:200]
        first = f[f.index("(") + 1:].split(",")[0]
        assert re.search(r'byref\(%"struct\.pac::vf64::Stage"\)', first), f[:300]
