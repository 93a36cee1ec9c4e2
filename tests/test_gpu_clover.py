"""The one-pass plaquette / clover kernel of SU(2) in d = 4 (su2_clover.hip) against
the oracle at the edges of its layout: partial blocks, the row wrap inside a
block, the longest row, extents of 1 to 3, a shorter last t-chunk; through
energy_density and the gradient-flow table, which takes every sum of it.

Sums of n terms of order one, compensated over blocks: a few 1e-16 relative per
partial, taken as 1e-12; the charge, a difference of such sums of size E V, as
1e-12 of E V."""
import numpy as np
import pytest

import su2_amd as S

pytestmark = pytest.mark.gpu
SEED = 13526463

DIMS = [(4, 4, 4, 4, 4), (2, 2, 2, 2, 4), (1, 3, 2, 1, 4), (3, 1, 5, 2, 4), (5, 9, 61, 3, 4),
        (3, 18, 15, 7, 4), (2, 3, 128, 5, 4), (8, 8, 8, 8, 4), (6, 33, 32, 9, 4),
        (2, 48, 48, 4, 4), (7, 24, 24, 13, 4)]


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("prec", [0, 1])
def test_energy_density_matches_oracle(oracle, dims, prec):
    U = oracle.hotstart(1, dims, SEED, 0.6)
    if prec == 1:
        U = U.astype(np.float32).astype(np.float64)
    V = dims[0] * dims[1] * dims[2] * dims[3]
    with S.Lattice(S.SU2, dims, 2.4, precision=prec) as lat:
        lat.set_links(U)
        for ss in (False, True):
            E, Q = lat.energy_density(ss=ss)
            E_ref, Q_ref = oracle.energy_density(1, dims, U, ss=ss)
            assert E == pytest.approx(E_ref, rel=1e-12, abs=1e-14)
            assert abs(Q - Q_ref) < 1e-12 * max(1.0, E_ref * V)


@pytest.mark.parametrize("dims", [(3, 18, 15, 7, 4), (8, 8, 8, 8, 4), (5, 6, 1, 7, 3)])
@pytest.mark.parametrize("group", [1, 0])
def test_flow_table_matches_oracle(oracle, dims, group):
    U = oracle.hotstart(group, dims, SEED, 0.6)
    _, ref = oracle.gradient_flow(group, dims, U.copy(), 2.4, 0.07, 0.01)
    with S.Lattice(group, dims, 2.4) as lat:
        lat.set_links(U)
        rows = lat.gradient_flow(0.07, 0.01)
        assert np.array_equal(lat.get_links(), U)
    assert rows.shape == ref.shape
    V = dims[0] * dims[1] * dims[2] * dims[3]
    # xi_R divides plaquette energies of a tenth of the plaquette itself
    assert np.abs(rows - ref).max() < 1e-11 * V ** 0.5
