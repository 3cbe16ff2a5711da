'''The rotational susceptibility at the edges of its state groups and sample counts per thread, against the oracle: one
state, a whole group, a padded one, more states than are staged at once; strips of one, two, four and eight samples per
thread. FP64 1e-10, FP32 1e-5 on the field (fixed steps).
'''
import pytest

from conftest import rel_l2
from searay_amd import configs, uppe_kernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nw,nr,n2,states', [(17, 8, 1, 12), (33, 8, 1, 3), (65, 16, 1, 10), (129, 8, 4, 11),
                                             (513, 8, 1, 70), (4097, 4, 1, 9)])
@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
def test_rotator_groups(oracle_mod, nw, nr, n2, states, precision):
    vol = configs.radial_raman_air(scale=max(1, 512 // (nw - 1)), steps=2, states=states)
    vol['wave grid'] = (nw, nr, n2, 2)
    vol['radial modes'] = nr
    print('rotator: %d states, strips of %d samples, %s' % (states - 2, 2 * (nw - 1), precision), flush=True)
    ref = uppe_kernel.track_with(vol, oracle_mod.oracle_factory)
    got = uppe_kernel.track_with(vol, uppe_kernel.hip_stepper_factory(precision))
    assert rel_l2(got[0][..., 1], ref[0][..., 1]) < (1e-10 if precision == 'fp64' else 1e-5)
    assert got[5] == ref[5]
