"""The shared-plaquette step (su2_md_plq.hpp) against the oracle at the sizes
where its layout can go wrong: rows that fill a block and rows that do not, the
row wrap inside a block, the longest row, extents of 1 and 2, a shorter last
t-chunk, the smallest volumes it takes, d = 3, anisotropic weights, and the
half-field layout ((16, 8, 8, 32), 3-volume a multiple of 256).

Tolerances: five force and four link sweeps with O(1) operands add some 20
roundings per sweep; FP64 20 * 9 * 2^-53 = 2e-14, taken as 1e-12 as for one
sweep elsewhere; FP32 (links and momenta rounded to 2^-24 per sweep) 20 * 9 *
2^-24 = 1.1e-5.  U(1) phases go up to 4 rather than 1: four times that."""
import numpy as np
import pytest

import su2_amd as S

pytestmark = pytest.mark.gpu
SEED = 13526463
TOL = {0: 1e-12, 1: 1.1e-5}

CASES = [  # Lx, Ly, Lz, Lt, nd, xi
    (16, 8, 8, 32, 4, 1.0), (16, 8, 8, 32, 4, 1.7), (5, 9, 61, 13, 4, 1.0),
    (3, 18, 15, 41, 4, 1.0), (1, 33, 32, 32, 4, 1.0), (2, 2, 64, 128, 4, 1.3),
    (33, 1, 31, 33, 4, 1.0), (20, 18, 2, 47, 4, 1.0), (59, 21, 1, 79, 3, 1.0),
    (40, 64, 1, 40, 3, 1.4), (7, 19, 31, 24, 4, 1.0), (8, 12, 48, 22, 4, 0.8),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("group", [1, 0])
def test_trajectory_matches_oracle(oracle, case, prec, group):
    *dims, xi = case
    dims = tuple(dims)
    if prec == 1 and dims[0] * dims[1] * dims[2] * dims[3] < 98304:
        # the FP32 form takes the step from 98304 sites
        dims = dims[:3] + (-(-98304 // (dims[0] * dims[1] * dims[2])),) + dims[4:]
    U0 = oracle.hotstart(group, dims, SEED, 0.4)
    P0 = oracle.initnormal(group, dims, SEED + 1)
    if prec == 1:
        U0 = U0.astype(np.float32).astype(np.float64)
        P0 = P0.astype(np.float32).astype(np.float64)
    U_ref, P_ref = oracle.integrate(group, dims, U0, P0.copy(), 2.4, S.OMF2, 2, tau=0.2, xi=xi)
    with S.Lattice(group, dims, 2.4, xi=xi, precision=prec) as lat:
        lat.set_links(U0)
        r = lat.md_trajectory(P0, S.OMF2, 2, tau=0.2)
        lat.md_finish(True)
        U, P = lat.get_links(), lat.get_momenta()
    tol = TOL[prec] * (1 if group == 1 else 4)
    assert np.abs(U - U_ref).max() < tol
    assert np.abs(P - P_ref).max() < 10 * tol  # momenta up to ~5, forces up to ~10
    # the step's own partial sums: kinetic energies and the start's action
    assert r["kin_old"] == pytest.approx(oracle.kinetic(group, dims, P0, compensated=True), rel=1e-13)
    assert r["kin_new"] == pytest.approx(oracle.kinetic(group, dims, P, compensated=True), rel=1e-13)
    assert r["gauge_old"] == pytest.approx(
        oracle.action(group, dims, U0, 2.4, xi=xi, compensated=True), rel=1e-13)


@pytest.mark.parametrize("dims", [(16, 8, 8, 32, 4), (5, 9, 61, 13, 4), (59, 21, 1, 79, 3)])
@pytest.mark.parametrize("group", [1, 0])
def test_momentum_only_and_zero_momentum_steps(oracle, dims, group):
    """The force alone (derivative), and the Runge-Kutta stages, whose first
    reads its momenta as zero (flat-gradient_flow.hh:17-50)."""
    U0 = oracle.hotstart(group, dims, SEED, 0.4)
    with S.Lattice(group, dims, 2.4) as lat:
        lat.set_links(U0)
        D = lat.derivative(1.0)
        lat.runge_kutta(0.01)
        W = lat.get_links()
    assert np.abs(D - oracle.derivative(group, dims, U0, 2.4)).max() < 1e-12
    assert np.abs(W - oracle.runge_kutta(group, dims, U0, 2.4, 0.01)).max() < 1e-12


def test_update_angles_beyond_the_series(oracle):
    """exp(eps P) with |eps P| from 0.3 to 3e3: the series below 1 and the
    reduced angle beyond it against the oracle's library functions.  The angle's
    own rounding, 2^-53 times its size, is in the bound."""
    dims = (16, 8, 8, 32, 4)
    U0 = oracle.coldstart(1, dims)
    P0 = oracle.initnormal(1, dims, SEED + 1)
    for scale in (0.2, 1.0, 30.0, 1000.0):
        P = scale * P0
        U_ref, _ = oracle.integrate(1, dims, U0, P.copy(), 1e-9, S.LEAPFROG, 1, tau=1.0)
        with S.Lattice(S.SU2, dims, 1e-9) as lat:
            lat.set_links(U0)
            lat.md_trajectory(P, S.LEAPFROG, 1, tau=1.0)
            lat.md_finish(True)
            U = lat.get_links()
        assert np.abs(U - U_ref).max() < 1e-15 * (4 + 10 * scale)
