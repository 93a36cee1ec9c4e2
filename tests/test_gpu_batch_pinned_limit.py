"""Downloads of batch members into pinned memory on both sides of the size up to which
the conversion kernel writes there itself (20 MiB) equal those into pageable memory
bit for bit, and write nothing beside them."""
import ctypes as C

import numpy as np
import pytest
import torch

import su2_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
def test_pinned_downloads_beside_the_limit(prec):
    dims = [(20, 20, 20, 20, 4), (20, 20, 20, 21, 4), (1024, 1, 1, 1280, 2), (1024, 1, 1, 1281, 2)]
    sizes = [d[0] * d[1] * d[2] * d[3] * (16 if d[4] == 4 else 2) * 8 for d in dims]
    assert [s <= 20 << 20 for s in sizes] == [True, False, True, False]
    members = [dict(group=S.SU2 if d[4] == 4 else S.U1, dims=d, beta=2.0, nsteps=1,
                    integrator="leapfrog") for d in dims]
    with S.Batch(members, precision=prec) as b:
        b.trajectory(1, metropolis=False)
        for i, s in enumerate(sizes):
            ref = b.get_links(i).reshape(-1)
            assert ref.size * 8 == s
            buf = torch.full((ref.size + 6,), 7.5, dtype=torch.float64, pin_memory=True)
            rc = b.lib.su2gpu_batch_get_links(
                b._h, i, C.cast(buf.data_ptr() + 24, C.POINTER(C.c_double)))
            assert rc == 0
            got = buf.numpy()
            assert np.array_equal(got[3:-3], ref)
            assert (got[:3] == 7.5).all() and (got[-3:] == 7.5).all()
