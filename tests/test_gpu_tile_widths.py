'''The exchange's tile widths and an autotuned batch's choice between them leave no trace in the result: members of a
batch too large for narrow tiles against standalone handles, which take them, bit for bit, with one source launch
shape for both. Modes that end inside a row tile, nonlinear bands that end inside a column tile, one and two row tiles
per wave (FP64), fixed and adaptive steps.
'''
import numpy as np
import pytest

from searay_amd import batch, configs, uppe_kernel

pytestmark = pytest.mark.gpu

# (frequencies, cells, modes, share of the band that is nonlinear, members)
GRIDS = [(257, 64, 51, 0.7, 10), (129, 256, 233, 1.0, 12)]


def _vol(nw, nr, nk, share, power, adaptive):
    vol = configs.radial_o2_ionization(scale=2048 // (nw - 1), nr=nr, steps=3, length='0.3 mm', power=power)
    vol['wave grid'] = (nw, nr, 1, 2)
    vol['radial modes'] = nk
    band = (0.0, max(2.0, vol['frequency band'][1]))
    vol['frequency band'] = band
    vol['nonlinear band'] = (0.0, max(1.4, share * band[1]))
    vol['minimum step'] = vol['size'][2] / vol['subcycles'] / (40 if adaptive else 1)
    return vol


@pytest.mark.parametrize('adaptive', [False, True])
@pytest.mark.parametrize('precision', ['fp64', 'fp32', 'bf16x3'])
@pytest.mark.parametrize('nw,nr,nk,share,members', GRIDS)
def test_autotuned_batch_equals_standalone(nw, nr, nk, share, members, precision, adaptive, monkeypatch):
    monkeypatch.setenv('SEARAY_UPPE_SOURCE_SPT', '2')
    monkeypatch.setenv('SEARAY_UPPE_WAVE_SOURCE', '0')
    vols = [_vol(nw, nr, nk, share, 0.5 + 0.2 * i, adaptive) for i in range(members)]
    print('tile widths: %d x %d x %d %s adaptive=%s' % (members, nw, nr, precision, adaptive), flush=True)
    with batch.Batch(vols, precision=precision, autotune=True) as b:
        b.set_fields()
        steps = b.advance()
        got = [m.get_state() for m in b.members]
        tiles = b.plan(0)['r2k']['tiles']
    for i in (0, members - 1):
        rs = uppe_kernel.RunSetup(vols[i])
        zi, _, length = rs.plane(0)
        with rs.make_stepper(uppe_kernel.hip_stepper_factory(precision)) as st:
            st.set_field(rs.stepper_field())
            n, _ = st.advance(zi, length, 0, rs.subcycles, rs.dzmin)
            want = st.get_state()
        assert n == steps[i]
        assert np.array_equal(got[i], want), (i, tiles, np.max(np.abs(got[i] - want)) / np.max(np.abs(want)))
