"""Downloads of batch members into pinned memory, which the conversion kernel
writes itself up to 4 MiB, equal those into pageable memory bit for bit: both
groups, a member above the limit, a destination inside a larger allocation, and
nothing written beside it."""
import ctypes as C

import numpy as np
import pytest
import torch

import su2_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
def test_pinned_download_equals_pageable(prec):
    members = [dict(group=S.U1, dims=(33, 1, 1, 17, 2), beta=2.0, nsteps=3),
               dict(group=S.SU2, dims=(5, 7, 1, 9, 3), beta=4.0, nsteps=3),
               dict(group=S.SU2, dims=(14, 14, 14, 14, 4), beta=2.3, nsteps=3)]  # 4.9 MB
    with S.Batch([dict(m, integrator="leapfrog") for m in members], precision=prec) as b:
        b.trajectory(1, metropolis=False)
        for i in range(len(members)):
            ref = b.get_links(i).reshape(-1)
            buf = torch.full((ref.size + 6,), 7.5, dtype=torch.float64, pin_memory=True)
            rc = b.lib.su2gpu_batch_get_links(
                b._h, i, C.cast(buf.data_ptr() + 24, C.POINTER(C.c_double)))
            assert rc == 0
            got = buf.numpy()
            assert np.array_equal(got[3:-3], ref)
            assert (got[:3] == 7.5).all() and (got[-3:] == 7.5).all()
