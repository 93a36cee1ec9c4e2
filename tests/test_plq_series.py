"""Errors of the sine and cosine series of the shared-plaquette step against 80-bit
arithmetic on the host (tests/native/plq_series_check.cpp), in units of 2^-53.

Derived bounds.  cos_sinc_fp64 up to x = 1: the last fused step rounds once, 1/2 ulp =
1/2 unit for results in [1/2, 1); what it adds to 1 is at most x / 2 with a relative error
of 1 1/2 units, 3/4 unit at x = 1, and the terms left out are below 0.1: 1.35, taken as
1.5 (a cosine series one power shorter leaves out 1.5 units alone).  Up to x = 12 the
root's half ulp is 2 units: 3.5 and, divided by a, 2.5.  Reduced sine and cosine of
angles up to 3e4: the reduced angle's rounding is half an ulp, the second part of pi/2
is rounded at 2^-87 and multiplied by up to 2^17: 1 1/2.  Beyond 1e5 the whole turns come
off with one more rounding of up to pi, 2 units: 3 1/2 (up to 4e14 here, where the angle's
own rounding is 2^49 units)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc"


def test_series_errors(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    exe = str(tmp_path / "plq_series_check")
    src = os.path.join(HERE, "native", "plq_series_check.cpp")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-x", "hip", src, "-o",
                    exe, "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"],
                   check=True, capture_output=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0
    c1, s1, c, s, rc, rs, fc, fs = map(float, out.stdout.split())
    assert c1 < 1.5 and s1 < 1.5, out.stdout
    assert c < 3.5 and s < 2.5 and rc < 1.5 and rs < 1.5, out.stdout
    assert fc < 3.5 and fs < 3.5, out.stdout
