'''The envelope source kernel with two samples per thread (strips of 128 to 2048 samples, fewer strips than CUs) and at
the lengths on either side, against the oracle: FP64 1e-10, FP32 1e-4 on the field (the paraxial tests' tolerances).
'''
import pytest

from conftest import rel_l2
from searay_amd import configs, paraxial_kernel, uppe_kernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nw', [64, 128, 512, 2048, 4096])
@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
def test_envelope_strip_lengths(oracle_mod, nw, precision):
    vol = configs.paraxial_air_filament(scale=16, steps=2, planes=20)
    vol['wave grid'] = (nw, 16, 1, 2)
    vol['radial modes'] = 11
    vol['size'] = vol['size'][:2] + (vol['size'][2] / 200,)
    print('envelope strips of %d samples %s' % (nw, precision), flush=True)
    ref = paraxial_kernel.track_with(vol, oracle_mod.oracle_factory)
    got = paraxial_kernel.track_with(vol, uppe_kernel.hip_stepper_factory(precision))
    assert rel_l2(got[0][..., 1], ref[0][..., 1]) < (1e-10 if precision == 'fp64' else 1e-4)
    assert got[5] == ref[5]
