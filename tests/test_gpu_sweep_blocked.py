"""The Metropolis sweep where its blocks walk t (Lt a multiple of 8, half a slice
a multiple of 256 sites) and next to that, against the oracle with the device's
visiting order and Philox stream: links within 1e-12 (every hit is some 50
roundings of O(1) operands, ten hits in a row 1e-13), and the same accepted
hits, also where nearly all (beta = 0.01) or few (beta = 40) are."""
import numpy as np
import pytest

import su2_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(8, 8, 8, 8, 4), (16, 8, 8, 16, 4), (8, 16, 4, 24, 4),
                                  (32, 32, 1, 16, 3), (8, 8, 8, 12, 4), (8, 8, 8, 9, 4)])
@pytest.mark.parametrize("group,beta", [(1, 0.01), (1, 2.4), (1, 40.0), (0, 1.0)])
def test_blocked_sweep_matches_oracle(oracle, dims, group, beta):
    U0 = oracle.hotstart(group, dims, 13526463, 0.7)
    U_ref, rates = oracle.sweep(group, dims, U0.copy(), beta, 987654321987, 5, 0.4, 10)
    with S.Lattice(group, dims, beta) as lat:
        lat.set_links(U0)
        got = lat.sweep(987654321987, 5, 0.4, 10)
        U = lat.get_links()
    assert got == pytest.approx(tuple(rates), abs=0, rel=1e-15)
    assert np.abs(U - np.asarray(U_ref)).max() < 1e-12
