"""The shared-plaquette step where its dispatch does not take it by itself
(SU2GPU_PLQ=1: wherever its layout applies), the momenta drawn inside its first step,
its instances with non-temporal accesses, and the switches that select between it and
the staple steps.  Switches are read once per process: child processes.

Tolerances of the trajectories are those of test_gpu_plq.py (the same steps)."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

import su2_amd as S

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SEED = 13526463
TOL = {0: 1e-12, 1: 1.1e-5}

_HEAD = r"""
import json, sys
import numpy as np
sys.path.insert(0, sys.argv[1])
import su2_amd as S
from oracle.oracle import Oracle
orc = Oracle()
SEED = 13526463
"""


def _child(code, env, *args):
    e = {k: v for k, v in os.environ.items() if not k.startswith("SU2GPU_")}
    e.update(env)
    out = subprocess.run([sys.executable, "-u", "-c", _HEAD + code, ROOT, *map(str, args)], env=e,
                         capture_output=True, text=True, timeout=110)
    print(env, out.stdout)
    assert out.returncode == 0, out.stdout + out.stderr
    return out.stdout


# rows that fill a block and rows that do not, the row wrap inside a block, the
# longest row, extents of 1 and 2, a shorter last chunk, planes of few sites, d = 3
CASES = [  # Lx, Ly, Lz, Lt, nd, xi
    (16, 8, 8, 8, 4, 1.0), (5, 9, 61, 3, 4, 1.0), (3, 18, 15, 7, 4, 1.7), (1, 33, 32, 5, 4, 1.0),
    (2, 2, 64, 9, 4, 1.3), (33, 1, 31, 6, 4, 1.0), (4, 1, 2, 5, 4, 1.0), (20, 18, 2, 7, 4, 1.0),
    (3, 3, 3, 3, 4, 0.8), (59, 21, 1, 9, 3, 1.0), (2, 8, 1, 33, 3, 1.4), (8, 12, 48, 5, 4, 0.8)]

# and, FP32 SU(2), walks of more than one slice
CASES32 = [(16, 8, 8, 96, 4, 1.7), (5, 9, 61, 36, 4, 1.0), (3, 18, 15, 122, 4, 1.0),
           (1, 33, 32, 94, 4, 1.0), (7, 19, 31, 24, 4, 1.0), (8, 12, 48, 22, 4, 0.8)]

_FORCED = r"""
for dims, xi, gps in json.loads(sys.argv[2]):
    dims = tuple(dims)
    for group, prec in gps:
        U0 = orc.hotstart(group, dims, SEED, 0.4)
        P0 = orc.initnormal(group, dims, SEED + 1)
        if prec == 1:
            U0 = U0.astype(np.float32).astype(np.float64)
            P0 = P0.astype(np.float32).astype(np.float64)
        U_ref, P_ref = orc.integrate(group, dims, U0, P0.copy(), 2.4, S.OMF2, 2, tau=0.2, xi=xi)
        with S.Lattice(group, dims, 2.4, xi=xi, precision=prec) as lat:
            lat.set_links(U0)
            r = lat.md_trajectory(P0, S.OMF2, 2, tau=0.2)
            lat.md_finish(True)
            U, P = lat.get_links(), lat.get_momenta()
        a = orc.action(group, dims, U0, 2.4, xi=xi, compensated=True)
        k = orc.kinetic(group, dims, P0, compensated=True)
        print("CASE", json.dumps([list(dims), group, prec, float(np.abs(U - U_ref).max()),
              float(np.abs(P - P_ref).max()), r["gauge_old"] / a - 1, r["kin_old"] / k - 1]), flush=True)
"""


def test_forced_step_matches_oracle():
    every = [(g, p) for g in (1, 0) for p in (0, 1)]
    cases = [(c[:5], c[5], every) for c in CASES] + [(c[:5], c[5], [(1, 1)]) for c in CASES32]
    out = _child(_FORCED, {"SU2GPU_PLQ": "1"}, json.dumps(cases))
    rows = [json.loads(ln[5:]) for ln in out.splitlines() if ln.startswith("CASE")]
    assert len(rows) == 4 * len(CASES) + len(CASES32)
    for dims, group, prec, du, dp, da, dk in rows:
        tol = TOL[prec] * (1 if group == 1 else 4)
        assert du < tol and dp < 10 * tol, (dims, group, prec, du, dp)
        # sums of 1e2 .. 1e5 terms, compensated: 1e-13; an action near zero cancels
        assert abs(da) < 1e-11 and abs(dk) < 1e-13, (dims, group, prec, da, dk)


_GEN = r"""
for group in (1, 0):
    for prec in (0, 1):
        for dims, xi in (((16, 8, 8, 16, 4), 1.0), ((5, 9, 12, 7, 4), 1.7), ((24, 10, 1, 9, 3), 1.0)):
            U = orc.hotstart(group, dims, 93, 0.5)
            with S.Lattice(group, dims, 2.4, xi=xi, precision=prec) as lat:
                lat.set_links(U)
                vals, fields = [], []
                for k in range(2):
                    r = lat.md_update(501 + k, S.OMF2, 6, momenta=S.MOMENTA_DEVICE)
                    vals += [r["kin_old"], r["kin_new"], r["gauge_old"], r["deltaH"]]
                    fields += [lat.get_links(), lat.get_momenta()]
            tag = "%d_%d_%d_%d" % (group, prec, dims[0], dims[4])
            np.savez(sys.argv[2] + tag + ".npz", vals=np.array(vals), **{"f%d" % i: f for i, f in enumerate(fields)})
            print("GEN", tag, flush=True)
"""


def test_momenta_drawn_in_the_first_step(tmp_path):
    """Device momenta drawn inside the first step against their own launch
    (SU2GPU_GENFUSE=0), both groups, both forms, d = 3 and 4.  The momenta are the same
    values; the first step's kernel is another instance of the same expressions, whose
    last bits may differ: FP64 as for a trajectory (1e-12 at tau = 0.2, times e^2 for tau =
    1), FP32 2^-24 per link and momentum up to 4, times the same growth and two
    trajectories: 6e-8 * 4 * 10 * 2 = 5e-6.  Kinetic energies of the drawn momenta: the
    same terms in the same order, 1e-12 at most."""
    tags = {}
    for v in ("1", "0"):
        base = str(tmp_path / f"gen{v}_")
        out = _child(_GEN, {"SU2GPU_PLQ": "1", "SU2GPU_GENFUSE": v}, base)
        tags[v] = [ln.split()[1] for ln in out.splitlines() if ln.startswith("GEN")]
    assert len(tags["1"]) == 12 and tags["1"] == tags["0"]
    for tag in tags["1"]:
        a, b = (np.load(str(tmp_path / f"gen{v}_{tag}.npz")) for v in ("1", "0"))
        tol = 1e-11 if tag.split("_")[1] == "0" else 5e-6
        for i in range(4):
            assert np.abs(a[f"f{i}"] - b[f"f{i}"]).max() < tol, (tag, i)
        va, vb = a["vals"].reshape(2, 4), b["vals"].reshape(2, 4)
        assert va[0, 0] == pytest.approx(vb[0, 0], rel=1e-12)
        np.testing.assert_allclose(va[:, 0], vb[:, 0], rtol=1e-12)  # the second draw's too
        # the first momenta and their energy are not trivial
        assert va[0, 0] > 0.1 * a["f1"].size


@pytest.mark.parametrize("group,dims,prec", [
    (0, (40, 42, 41, 42, 4), 0), (0, (58, 57, 56, 32, 4), 1), (1, (101, 100, 1, 104, 3), 0),
    (0, (156, 157, 1, 156, 3), 0), (1, (128, 129, 1, 127, 3), 1)])
def test_non_temporal_instances(oracle, group, dims, prec):
    """Fields beyond 256 MB: the instances with non-temporal stores and momentum loads,
    U(1) and d = 3.  One leapfrog step against the oracle."""
    V = dims[0] * dims[1] * dims[2] * dims[3]
    assert dims[4] * V * (11 if group else 3) * (8 if prec == 0 else 4) > 256 << 20
    U0 = oracle.hotstart(group, dims, SEED, 0.4)
    P0 = oracle.initnormal(group, dims, SEED + 1)
    if prec == 1:
        U0 = U0.astype(np.float32).astype(np.float64)
        P0 = P0.astype(np.float32).astype(np.float64)
    U_ref, P_ref = oracle.integrate(group, dims, U0, P0.copy(), 2.4, S.LEAPFROG, 1, tau=0.1)
    with S.Lattice(group, dims, 2.4, precision=prec) as lat:
        lat.set_links(U0)
        lat.md_trajectory(P0, S.LEAPFROG, 1, tau=0.1)
        lat.md_finish(True)
        U, P = lat.get_links(), lat.get_momenta()
    tol = TOL[prec] * (1 if group == 1 else 4)
    assert np.abs(U - U_ref).max() < tol
    assert np.abs(P - P_ref).max() < 10 * tol


_BITS = r"""
dims = (16, 8, 8, 32, 4)
U = orc.hotstart(1, dims, 91, 0.5)
P = orc.initnormal(1, dims, 92)
with S.Lattice(1, dims, 2.4) as lat:
    lat.set_links(U)
    lat.md_trajectory(P, S.OMF2, 4)
    lat.md_finish(True)
    np.save(sys.argv[2], lat.get_links())
"""


def test_switches_select_the_step(tmp_path):
    """The two steps round differently, so the bits of a trajectory show which one ran:
    by itself the 32768 sites of this lattice take the shared-plaquette step, and a set
    switch of the staple steps selects those."""
    got = {}
    for name, env in (("auto", {}), ("plq", {"SU2GPU_PLQ": "1"}), ("staple", {"SU2GPU_PLQ": "0"}),
                      ("tw", {"SU2GPU_TW": "1"}), ("nt", {"SU2GPU_NT": "0"}),
                      ("both", {"SU2GPU_TW": "1", "SU2GPU_PLQ": "1"})):
        f = str(tmp_path / (name + ".npy"))
        _child(_BITS, env, f)
        got[name] = np.load(f)
    same = lambda a, b: np.array_equal(got[a], got[b])  # noqa: E731
    assert not same("plq", "staple") and np.abs(got["plq"] - got["staple"]).max() < 1e-11
    assert same("auto", "plq") and same("both", "plq")
    assert same("tw", "staple") and same("nt", "staple")
