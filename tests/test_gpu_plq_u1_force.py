"""The FP64 U(1) force of the shared-plaquette step keeps the precision of the staple
steps, which sum three phases, take the sine and cosine, sum the staples and multiply
by the link.  That arithmetic is replayed here on the host, and the step's rms error
against the force in 80 bits may exceed the replay's by 5 %: 131072 components know
the rms to 0.3 %, and the device contracts products that the replay rounds.  With the
plaquette's angle from three plain differences it is 12 % above."""
import numpy as np
import pytest

import su2_amd as S

pytestmark = pytest.mark.gpu


def _force(U, dims, T):
    """Im(exp(i U) K), the staple steps' operations in type T: (V nd,)"""
    Lx, Ly, Lz, Lt, nd = dims
    shape = (Lt, Lx, Ly, Lz)[:nd]
    q = [U.reshape(shape + (nd,))[..., m].astype(T) for m in range(nd)]
    up = lambda a, d: np.roll(a, -1, d)  # noqa: E731
    dn = lambda a, d: np.roll(a, 1, d)  # noqa: E731
    out = []
    for mu in range(nd):
        re = im = T(0)
        for nu in range(nd):
            if nu != mu:
                a = (up(q[nu], mu) - up(q[mu], nu)) - q[nu]
                b = dn((-up(q[nu], mu) - q[mu]) + q[nu], nu)
                re = (re + np.cos(a)) + np.cos(b)
                im = (im + np.sin(a)) + np.sin(b)
        out.append(np.cos(q[mu]) * im + np.sin(q[mu]) * re)
    return np.stack(out, -1).ravel()


@pytest.mark.parametrize("dims", [(16, 8, 16, 16, 4), (48, 32, 1, 32, 3)])
def test_u1_force_error(dims):
    V = dims[0] * dims[1] * dims[2] * dims[3]
    U = np.random.RandomState(3).randn(V * dims[4]) * 1.2
    exact = _force(U, dims, np.longdouble)
    want = (_force(U, dims, np.float64) - exact).astype(np.float64)
    with S.Lattice(S.U1, dims, 1.0) as lat:
        lat.set_links(U)
        got = (lat.derivative(1.0).ravel() - exact).astype(np.float64)
    rms = lambda x: float(np.sqrt((x * x).mean()))  # noqa: E731
    print(dims, "rms error", rms(got), "replay", rms(want))
    assert rms(got) < 1.05 * rms(want)
