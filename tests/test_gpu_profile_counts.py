"""su2gpu_profile_read counts the launches of a name: one of energy_density for one call,
on lattices that take the fused plaquette and clover pass and on those that do not."""
import pytest

import su2_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("group,dims", [(1, (8, 8, 8, 8, 4)), (1, (8, 6, 1, 4, 3)), (0, (6, 4, 4, 8, 4)),
                                        (1, (4, 4, 4, 4, 4)), (0, (8, 1, 1, 8, 2))])
def test_one_launch_counted_once(group, dims):
    with S.Lattice(group, dims, 2.0) as lat:
        lat.hotstart(7, 0.5)
        lat.profile(True)
        for clover in (True, False):
            for ss in (False, True):
                lat.profile_reset()
                lat.energy_density(clover=clover, ss=ss)
                assert lat.profile_read("energy_density")[1] == 1, (clover, ss)
