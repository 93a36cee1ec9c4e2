"""Which lattices the dispatch gives to the shared-plaquette step: enough sites, and planes
that do not leave most lanes idle.  The two steps round differently, so the bits of a
trajectory show which one ran (switches are read once per process: child processes).
The two steps' difference: the tolerances of test_gpu_plq.py for each, times the longer
trajectory."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOL = {0: 1e-12, 1: 1.1e-5}

_ROUTES = [  # group, precision, dims, takes it
    (1, 0, (16, 8, 8, 32, 4), True), (1, 0, (32, 9, 9, 14, 4), True), (1, 0, (64, 3, 3, 64, 4), False),
    (1, 0, (64, 4, 4, 34, 4), False), (1, 0, (24, 24, 1, 60, 3), True), (1, 0, (8, 16, 16, 15, 4), False),
    (1, 1, (24, 24, 22, 13, 4), True), (1, 1, (18, 18, 18, 18, 4), False),
    (1, 1, (64, 6, 6, 64, 4), False), (1, 1, (48, 48, 1, 48, 3), True),
    (0, 0, (32, 5, 6, 40, 4), True), (0, 0, (64, 4, 4, 64, 4), False),
    (0, 1, (32, 9, 9, 40, 4), True), (0, 1, (32, 5, 6, 110, 4), False)]

_CHILD = r"""
import json, sys
import numpy as np
sys.path.insert(0, sys.argv[1])
import su2_amd as S
from oracle.oracle import Oracle
orc = Oracle()
for group, prec, dims, _ in json.loads(sys.argv[3]):
    dims = tuple(dims)
    U = orc.hotstart(group, dims, 91, 0.5)
    P = orc.initnormal(group, dims, 92)
    with S.Lattice(group, dims, 2.4, precision=prec) as lat:
        lat.set_links(U)
        lat.md_trajectory(P, S.OMF2, 3, tau=0.5)
        lat.md_finish(True)
        np.save(sys.argv[2] + "_".join(map(str, (group, prec) + dims)) + ".npy", lat.get_links())
    print("ROUTE", group, prec, dims, flush=True)
"""


def test_dispatch_takes_the_step_where_it_is_faster(tmp_path):
    got = {}
    for name in ("auto", "1", "0"):
        e = {k: v for k, v in os.environ.items() if not k.startswith("SU2GPU_")}
        if name != "auto":
            e["SU2GPU_PLQ"] = name
        base = str(tmp_path / (name + "_"))
        out = subprocess.run([sys.executable, "-u", "-c", _CHILD, ROOT, base, json.dumps(_ROUTES)],
                             env=e, capture_output=True, text=True, timeout=110)
        print(name, out.stdout)
        assert out.returncode == 0, out.stdout + out.stderr
        got[name] = [np.load(base + "_".join(map(str, r[:2] + r[2])) + ".npy") for r in _ROUTES]
    for i, (group, prec, dims, takes) in enumerate(_ROUTES):
        d = np.abs(got["1"][i] - got["0"][i]).max()
        assert 0 < d < 40 * TOL[prec], (group, prec, dims, d)
        assert np.array_equal(got["auto"][i], got["1" if takes else "0"][i]), (group, prec, dims)
