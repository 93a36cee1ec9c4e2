"""Batches whose SU(2) d = 4 members together pass the line of the shared-plaquette
ticks (32768 sites in FP64, 98304 in FP32) against single-lattice handles, which
take other kernels for most of these extents: rows of one block and of several,
ragged last blocks, chunks that do not divide t, members that end on every kind of
tick, and a rest below the line that goes back to the link tiles.

Tolerance: the forms differ by rounding alone, 40 operations a step on links of
size 1 over at most 24 steps of a chaotic but short trajectory (tau = 1, growth below
e^2): FP64 24 * 40 * 1e-16 * 8 < 1e-10; FP32 24 * 8 roundings of 6e-8 * 8 (sums are
FP64) < 1e-4, of which links at rest in a normalised form keep a fifth: 2e-5.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SEED = 13526463

# small members end last, so that the rest falls below the line
SMALL = [
    dict(group=1, dims=(3, 5, 9, 7, 4), beta=2.3, integrator="omf2", nsteps=12),
    dict(group=1, dims=(8, 8, 8, 8, 4), beta=2.5, integrator="leapfrog", nsteps=20),
    dict(group=1, dims=(2, 21, 12, 5, 4), beta=2.4, integrator="omf2", nsteps=4),
    dict(group=1, dims=(12, 12, 12, 13, 4), beta=2.4, integrator="leapfrog", nsteps=9),
    dict(group=1, dims=(16, 16, 16, 11, 4), beta=2.4, integrator="leapfrog", nsteps=10),
    dict(group=0, dims=(6, 1, 1, 5, 2), beta=1.5, integrator="leapfrog", nsteps=4),
    dict(group=1, dims=(9, 8, 1, 11, 3), beta=4.0, integrator="omf2", nsteps=3),
]
LARGE = SMALL + [dict(group=1, dims=(16, 16, 16, 16, 4), beta=2.4, integrator="omf2", nsteps=4)]


@pytest.fixture(scope="module")
def S():
    import su2_amd
    su2_amd.load_library()
    return su2_amd


@pytest.mark.parametrize("prec,members,graph", [(0, SMALL, False), (0, SMALL, True), (1, LARGE, False),
                                                (1, SMALL, False)],
                         ids=["fp64", "fp64-graph", "fp32", "fp32-below"])
def test_members_match_single_lattices(S, oracle, prec, members, graph):
    starts = [(oracle.hotstart(m["group"], m["dims"], SEED + i, 0.4),
               oracle.initnormal(m["group"], m["dims"], SEED + 50 + i)) for i, m in enumerate(members)]
    with S.Batch(members, precision=prec) as b:
        b.use_graph(graph)
        for rep in range(3 if graph else 1):
            for i, (U, P) in enumerate(starts):
                b.set_links(i, U)
                b.set_momenta(i, P)
            res = b.trajectory(0, momenta=S.MOMENTA_HOST, metropolis=False)
            got = [b.get_links(i) for i in range(len(members))]
            if rep:
                for x, y in zip(got, first):
                    np.testing.assert_array_equal(x, y)
            first = got
    for i, m in enumerate(members):
        U, P = starts[i]
        with S.Lattice(m["group"], m["dims"], m["beta"], precision=prec) as lat:
            lat.set_links(U)
            r = lat.md_trajectory(P, S.INTEGRATORS[m["integrator"]], m["nsteps"])
            lat.md_finish(True)
            want = lat.get_links()
        np.testing.assert_allclose(got[i], want, atol=1e-10 if prec == 0 else 2e-5,
                                   err_msg=f"member {i} {m['dims']}")
        assert res[i]["deltaH"] == pytest.approx(r["deltaH"], rel=1e-9 if prec == 0 else 1e-3,
                                                 abs=1e-9 if prec == 0 else 5e-3)
