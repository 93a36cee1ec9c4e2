"""One-pass stages of the gradient-flow adjoint (FP32, SU(2), d = 4) against the
FP64 two-pass form, which tests/test_gpu_flow.py pins by finite differences.

Tolerance: a component of the cotangent goes through at most 128 roundings of half
an ulp in one stage (six planes of four products on either side of the neighbour
sums, the Taylor series, and the forward stage's own link), each relative to the
largest component, so 3 n stages stay within 3 n 128 2^-24 of it.  At eps = 1, where
|A| > 1 takes the general branch, a stage's Jacobian reaches a norm of about 5 and
three of them amplify an early rounding by about 100.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SEED = 13526463


@pytest.fixture(scope="module")
def S():
    import su2_amd
    su2_amd.load_library()
    return su2_amd


@pytest.mark.parametrize("dims,xi,nsteps,ckpt,obs,eps", [
    ((2, 2, 2, 2, 4), 1.0, 3, 2, 0, 0.02),      # every neighbour wraps, one wavefront
    ((3, 1, 1, 5, 4), 1.0, 2, 1, 1, 0.02),      # a block of one row, its own neighbour
    ((1, 2, 7, 3, 4), 1.0, 2, 3, 0, 0.02),      # one slice
    ((5, 3, 33, 10, 4), 1.0, 4, 3, 0, 0.02),    # several row blocks, a ragged last one
    ((4, 2, 3, 65, 4), 1.4, 5, 2, 1, 0.02),     # a row of more than a wavefront, weights
    ((2, 2, 3, 128, 4), 1.0, 2, 2, 0, 0.02),    # the longest row
    ((2, 2, 3, 129, 4), 1.0, 2, 2, 0, 0.02),    # one more: the two-pass form
    ((9, 4, 16, 16, 4), 1.0, 1, 1, 0, 1.0),     # |A| > 1
])
def test_one_pass_stage_against_fp64(S, oracle, dims, xi, nsteps, ckpt, obs, eps):
    U = oracle.random_gauge_trafo(1, dims, oracle.hotstart(1, dims, SEED, 0.6), 654321)
    U = U.astype(np.float32).astype(np.float64)
    g = []
    for prec in (S.FP64, S.FP32):
        with S.Lattice(S.SU2, dims, 2.4, xi=xi, precision=prec) as lat:
            lat.set_links(U)
            lat.flow_forward(eps, nsteps, ckpt, obs)
            g.append(lat.flow_backward())
    tol = 3 * nsteps * 128 * 2.0 ** -24 * (100 if eps > 0.5 else 1)
    assert np.abs(g[1] - g[0]).max() <= tol * np.abs(g[0]).max()
