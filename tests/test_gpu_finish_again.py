'''Reading a field with its diagnostics leaves nothing behind: the same run afterwards, with and without diagnostics, gives
the same bits as before.
'''
import numpy as np
import pytest

from searay_amd import configs, paraxial_kernel, uppe_kernel

pytestmark = pytest.mark.gpu


def _setup(model):
    if model == 'radial':
        vol = configs.radial_o2_ionization(scale=8, nr=16, steps=4, length='0.3 mm')
        vol['nonlinear band'] = (0.0, 0.6 * vol['frequency band'][1])
        return uppe_kernel.RunSetup(vol)
    if model == 'cartesian':
        vol = configs.cartesian_filamentation(scale=8, steps=100)
        vol['wave grid'] = (33, 8, 4, 2)
        return uppe_kernel.RunSetup(vol)
    vol = configs.paraxial_air_filament(scale=4, planes=20)
    return paraxial_kernel.RunSetup(vol)


@pytest.mark.parametrize('model', ['radial', 'cartesian', 'envelope'])
@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
def test_runs_after_diagnostics(model, precision):
    print('finish and run again: %s %s' % (model, precision), flush=True)
    rs = _setup(model)
    zi, _, length = rs.plane(0)
    with rs.make_stepper(uppe_kernel.hip_stepper_factory(precision)) as st:
        runs = []
        for diagnostics in (True, True, False):
            st.set_field(rs.stepper_field())
            st.advance(zi, length, 0, rs.subcycles, rs.dzmin, max_steps=3)
            q = st.get_state()
            runs.append((q, st.finish(length, want_diagnostics=diagnostics)))
    assert np.linalg.norm(runs[0][1][1]) > 0
    for q, out in runs[1:]:
        assert np.array_equal(q, runs[0][0])
        for a, b in zip(out, runs[0][1]):
            assert a is None or np.array_equal(a, b)
