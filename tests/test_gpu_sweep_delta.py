"""Metropolis hits of a width whose angle makes many turns: 2 delta u half turns beyond
2^31 of them.  At beta = 0 every hit is accepted, so the links are the drawn elements.

The angle 2 pi delta u of the oracle is rounded to 2^-53 of its size, 2^31 * 2 pi * 2^-53
= 1.5e-6, and its product with pi as much again: 1e-5."""
import numpy as np
import pytest

import su2_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("delta", [0.4, 2.0 ** 20, -3.0 * 2.0 ** 20, 2.0 ** 31])
def test_wide_hits_match_oracle(oracle, delta):
    dims = (8, 4, 6, 4, 4)
    U0 = oracle.coldstart(1, dims)
    U_ref, _ = oracle.sweep(1, dims, U0.copy(), 0.0, 99, 3, delta, 1)
    with S.Lattice(S.SU2, dims, 0.0) as lat:
        lat.set_links(U0)
        rate = lat.sweep(99, 3, delta, 1)
        U = lat.get_links()
    assert rate == (1.0, 1.0)
    assert np.abs(U - np.asarray(U_ref)).max() < 1e-5
