"""The Metropolis sweep's order of blocks in groups of t slices (Lt a multiple of 8, half
a slice a multiple of 256 sites): slices per XCD that fall into groups of 4, 5, 6, 7, 3
and 1, one block and several per slice, d = 2, 3, 4, against the oracle with the
device's visiting order and Philox stream.  Links within 1e-12 (two hits of some 50
roundings of O(1) operands) and the same accepted hits."""
import numpy as np
import pytest

import su2_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(8, 8, 8, 64, 4), (8, 8, 8, 40, 4), (16, 8, 8, 48, 4),
                                  (8, 8, 8, 56, 4), (8, 8, 8, 72, 4), (8, 8, 8, 88, 4),
                                  (16, 32, 1, 128, 3), (32, 32, 1, 80, 3), (512, 1, 1, 128, 2)])
def test_grouped_sweep_matches_oracle(oracle, dims):
    for group, beta in ((1, 2.4), (0, 1.0)):
        U0 = oracle.hotstart(group, dims, 13526463, 0.7)
        U_ref, rates = oracle.sweep(group, dims, U0.copy(), beta, 987654321987, 5, 0.4, 2)
        with S.Lattice(group, dims, beta) as lat:
            lat.set_links(U0)
            got = lat.sweep(987654321987, 5, 0.4, 2)
            U = lat.get_links()
        assert got == pytest.approx(tuple(rates), abs=0, rel=1e-15)
        assert np.abs(U - np.asarray(U_ref)).max() < 1e-12
