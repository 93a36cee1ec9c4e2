"""Launch layout of the shared-plaquette step, replayed on the host
(tests/native/plq_layout_check.cpp): every site exactly once, periodic
neighbours, LDS partners."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc"

# d, (t, x, y, z), resident blocks per CU: rows that fill a block and rows that do not,
# extents of 1 to 3 (a neighbour in both directions), one block per plane (the
# row wrap inside the block), chunks that divide Lt and a shorter last chunk
CASES = [
    (4, (8, 4, 32, 32), 3), (4, (27, 20, 18, 15), 3), (4, (12, 6, 24, 24), 3),
    (4, (7, 3, 48, 48), 1), (4, (4, 4, 4, 4), 3), (4, (2, 2, 2, 2), 3),
    (4, (1, 1, 1, 2), 3), (4, (3, 1, 2, 64), 1), (4, (5, 2, 40, 40), 2),
    (4, (5, 2, 3, 128), 2), (4, (16, 3, 5, 3), 1), (4, (9, 2, 7, 61), 3), (3, (21, 16, 16, 1), 3),
    (3, (79, 21, 59, 1), 8), (3, (3, 2, 64, 1), 4), (3, (8, 5, 3, 1), 8),
]


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    exe = str(tmp_path_factory.mktemp("plq") / "plq_layout_check")
    src = os.path.join(HERE, "native", "plq_layout_check.cpp")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-x", "hip", src, "-o",
                    exe, "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"],
                   check=True, capture_output=True)
    return exe


@pytest.mark.parametrize("nd,ext,slots", CASES)
def test_every_site_once_with_its_neighbours(check, nd, ext, slots):
    out = subprocess.run([check, str(nd), *map(str, ext), str(slots)], capture_output=True,
                         text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.startswith("ok"), (out.returncode, out.stdout)


def test_not_applicable_geometries(check):
    # a row longer than the longest taken, a row of one site
    for ext in ((4, 4, 4, 129), (4, 4, 4, 1)):
        out = subprocess.run([check, "4", *map(str, ext), "2"], capture_output=True, text=True)
        assert out.returncode == 0 and out.stdout.startswith("not applicable")
