"""The library's scratch arena and block pool on the CPU, over a stand-in HIP
runtime whose allocations fail on request
(baby_shark_amd/csrc/alloc_check.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc compiles the host code")


def test_allocation_failures_leave_nothing_behind():
    csrc = os.path.join(ROOT, "baby_shark_amd", "csrc")
    for cmd in (["make", "-s", "-C", csrc, "alloc_check"], [os.path.join(csrc, "_build", "alloc_check")]):
        r = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
        assert r.returncode == 0, f"{cmd}: {r.returncode}\n{r.stdout[-2000:]}\n{r.stderr[-4000:]}"
    assert "allocation checks passed" in r.stdout
