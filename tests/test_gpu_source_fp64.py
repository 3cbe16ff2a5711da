'''The FP64 source kernel's instances for one strip length each (128 to 4096 samples) and the lengths on either side,
with few strips (wide workgroups) and with as many as CUs, in ionising gas at fields from the rate's cutoff to well
above it, against the oracle: 1e-10 on the field, the same steps.
'''
import pytest

from conftest import rel_l2
from searay_amd import configs, uppe_kernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nw,nr,power', [(33, 8, 2.0), (65, 8, 2.0), (129, 8, 2.0), (129, 256, 2.0), (257, 8, 1e-6),
                                         (513, 8, 4.0), (513, 256, 1.0), (1025, 8, 2.0), (2049, 8, 2.0),
                                         (4097, 4, 2.0)])
@pytest.mark.parametrize('rate', ['explicit', 'series'])
def test_source_fp64_lengths(oracle_mod, nw, nr, power, rate):
    vol = configs.radial_o2_ionization(scale=max(1, 2048 // (nw - 1)), nr=nr, steps=2, length='0.2 mm', power=power,
                                       rate=rate)
    vol['wave grid'] = (nw, nr, 1, 2)
    vol['radial modes'] = nr
    vol['frequency band'] = (0.0, max(2.0, vol['frequency band'][1]))
    vol['nonlinear band'] = (0.0, vol['frequency band'][1])
    print('FP64 strips of %d samples, %d of them, %s' % (2 * (nw - 1), nr, rate), flush=True)
    ref = uppe_kernel.track_with(vol, oracle_mod.oracle_factory)
    got = uppe_kernel.track_with(vol, uppe_kernel.hip_stepper_factory('fp64'))
    assert rel_l2(got[0][..., 1], ref[0][..., 1]) < 1e-10
    assert got[5] == ref[5]
