"""The plan of the shared-plaquette step on the host (tests/native/plq_plan_check.cpp): the
chunk choice equals a plain sum over the rounds and takes microseconds also for a lattice
long in t (it is made at every launch: 30 us for 2^20 slices; 1 ms is the bound, the plain
sum takes 6), and the share of lanes in use."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc"


def test_plan(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    exe = str(tmp_path / "plq_plan_check")
    src = os.path.join(HERE, "native", "plq_plan_check.cpp")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-x", "hip", src, "-o",
                    exe, "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"],
                   check=True, capture_output=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and "ok" in out.stdout, (out.returncode, out.stdout)
