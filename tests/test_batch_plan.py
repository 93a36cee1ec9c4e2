"""Which ticks of a batch's SU(2) d = 4 members run on shared-plaquette tiles
(plan_batch_plq, tests/native/batch_plan_check.cpp): the batches of
test_gpu_batch_plq.py do, with a plan made anew and a rest on the link tiles, and a
member that the layout does not take keeps the others from it only while it runs."""
import os
import subprocess

import pytest

from test_gpu_batch_plq import LARGE, SMALL

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    exe = str(tmp_path_factory.mktemp("batch") / "batch_plan_check")
    src = os.path.join(HERE, "native", "batch_plan_check.cpp")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-I",
                    os.path.join(HERE, "..", "include"), "-x", "hip", src, "-o", exe, "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops"], check=True, capture_output=True)

    def run(prec, members):
        """[(plan, tiles, running sites)] of every tick"""
        args = [str(prec)]
        for dims, npairs in members:
            args += [str(v) for v in dims[:4]] + [str(npairs)]
        out = subprocess.run([exe] + args, capture_output=True, text=True, timeout=60)
        assert out.returncode == 0, (out.returncode, out.stdout)
        return [tuple(map(int, ln.split()[1:])) for ln in out.stdout.splitlines()]
    return run


def _d4(members):
    return [(m["dims"], m["nsteps"] * (2 if m["integrator"] == "omf2" else 1)) for m in members
            if m["group"] == 1 and m["dims"][4] == 4]


def test_gpu_test_batches_run_on_plaquette_tiles(plan):
    for prec, members, plans in ((0, SMALL, 2), (1, LARGE, 1)):
        ticks = plan(prec, _d4(members))
        line = 32768 if prec == 0 else 98304
        assert [p >= 0 for p, _, _ in ticks] == [run >= line for _, _, run in ticks]
        assert ticks[0][0] == 0 and ticks[-1][0] == -1
        assert max(p for p, _, _ in ticks) + 1 >= plans
    assert all(p < 0 for p, _, _ in plan(1, _d4(SMALL)))


def test_member_outside_the_layout_counts_only_while_it_runs(plan):
    rest = [((16, 16, 16, 16), 30), ((16, 16, 16, 16), 25), ((8, 8, 8, 8), 20)]
    for odd in ((4, 4, 129, 4), (6, 6, 1, 6)):
        ticks = plan(1, rest + [(odd, 10)])
        assert [p >= 0 for p, _, _ in ticks] == [False] * 11 + [True] * 15 + [False] * 5
    # planes that leave three quarters of the lanes idle likewise
    ticks = plan(0, rest + [((16, 4, 4, 256), 12)])
    assert [p >= 0 for p, _, _ in ticks] == [False] * 13 + [True] * 18


def test_lanes_to_a_site(plan):
    # three quarters of the lanes: FP64 takes them, FP32 does not
    assert plan(0, [((12, 12, 12, 12), 5)] * 8)[0][0] == 0
    assert plan(1, [((12, 12, 12, 12), 5)] * 8)[0][0] == -1
    assert plan(1, [((8, 8, 8, 8), 5)] * 32)[0][0] == 0
