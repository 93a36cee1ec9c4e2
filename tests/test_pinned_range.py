"""Which host ranges a batch download may be written to by a kernel
(tests/native/pinned_range_check.cpp): whole ranges of one pinned allocation only."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc"


def test_only_ranges_of_one_pinned_allocation(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    exe = str(tmp_path / "pinned_range_check")
    src = os.path.join(HERE, "native", "pinned_range_check.cpp")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-x", "hip", src, "-o",
                    exe], check=True, capture_output=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.startswith("ok"), (out.returncode, out.stdout)
