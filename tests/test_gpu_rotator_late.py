'''A rotator loaded into a handle or a batch that has stepped without one (another launch shape of the source kernel), and
taken out again: the states of handles that had it, or had none, from the start. Each step call starts from the same field,
so equal launch shapes give equal bits.
'''
import numpy as np
import pytest

from searay_amd import batch, configs, paraxial_kernel, uppe_kernel

pytestmark = pytest.mark.gpu


def _vol(model, rotator):
    if model == 'envelope':
        vol = configs.paraxial_air_filament(scale=2, planes=20, rotator_states=32 if rotator else 0)
        vol['wave grid'] = (128, 16, 1, 20)
        vol['radial modes'] = 11
        return vol
    vol = configs.radial_kerr_air(scale=4, steps=4)
    if rotator:
        vol['rotator'] = configs.n2_rotator(32)
    vol['wave grid'] = (129, 16, 1, 2)
    vol['radial modes'] = 13
    return vol


def _advance(rs, st):
    zi, _, length = rs.plane(0)
    st.set_field(rs.stepper_field())
    st.advance(zi, length, 0, rs.subcycles, rs.dzmin, max_steps=3)
    return st.get_state()


@pytest.mark.parametrize('model', ['envelope', 'uppe'])
@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
def test_rotator_after_steps(model, precision):
    print('rotator after steps: %s %s' % (model, precision), flush=True)
    module = paraxial_kernel if model == 'envelope' else uppe_kernel
    make = uppe_kernel.hip_stepper_factory(precision)
    with_rot, without = module.RunSetup(_vol(model, True)), module.RunSetup(_vol(model, False))
    with with_rot.make_stepper(make) as st:
        want = _advance(with_rot, st)
    dt = with_rot.dt if model == 'uppe' else paraxial_kernel.source_dt(with_rot.mat.w)
    with without.make_stepper(make) as st:
        plain = _advance(without, st)
        st.set_rotator(with_rot.rotator, dt)
        assert np.array_equal(_advance(without, st), want)
        st.set_rotator(None, dt)
        assert np.array_equal(_advance(without, st), plain)
    assert not np.array_equal(plain, want)


@pytest.mark.parametrize('autotune', [False, True])
def test_rotator_after_batch_steps(autotune):
    vols = [_vol('uppe', False) for _ in range(3)]
    rotator, dt = configs.n2_rotator(32), uppe_kernel.RunSetup(vols[0]).dt

    def steps(b):
        b.set_fields()
        b.advance(max_steps=3)
        return [m.get_state() for m in b.members]

    print('rotator after batch steps, autotune %s' % autotune, flush=True)
    with batch.Batch([_vol('uppe', True) for _ in range(3)], precision='fp64', autotune=False) as b:
        want = steps(b)
    with batch.Batch(vols, precision='fp64', autotune=autotune) as b:
        steps(b)
        for m in b.members:
            m.set_rotator(rotator, dt)
        got = steps(b)
    for g, w in zip(got, want):
        assert np.allclose(g, w, rtol=0, atol=1e-12 * np.max(np.abs(w)))
