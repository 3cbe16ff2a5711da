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


@pytest.mark.parametrize('precision', ['fp64', 'fp32', 'bf16x3'])
def test_untuned_batches_plan_for_all_instances(precision):
    nw, nr, nk, share, members = GRIDS[0]
    vols = [_vol(nw, nr, nk, share, 0.5, False) for _ in range(members)]
    f1 = int(np.nonzero(uppe_kernel.RunSetup(vols[0]).nl_filter)[0][-1]) + 1
    tiles = []
    for n in (2, members):
        print('tiles of %d x %d x %d %s' % (n, nw, nr, precision), flush=True)
        with batch.Batch(vols[:n], precision=precision, autotune=False) as b:
            b.set_fields()
            b.advance(max_steps=1)
            tiles.append(b.plan(0)['r2k']['tiles'])
    assert tiles == [(f1 + 3) // 4, (f1 + 7) // 8]


@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
@pytest.mark.parametrize('adaptive', [False, True])
@pytest.mark.parametrize('nw,nr,nk,share,members', GRIDS)
def test_exchange_equals_separate_contractions(nw, nr, nk, share, members, precision, adaptive, monkeypatch):
    rs = uppe_kernel.RunSetup(_vol(nw, nr, nk, share, 1.0, adaptive))
    zi, _, length = rs.plane(0)
    states = []
    for width in (None, '8'):  # a pinned width asks for the separate contractions
        if width:
            monkeypatch.setenv('SEARAY_UPPE_TILE_WIDTH', width)
        print('exchange or not: %d x %d %s width %s' % (nw, nr, precision, width), flush=True)
        with rs.make_stepper(uppe_kernel.hip_stepper_factory(precision)) as st:
            st.set_field(rs.stepper_field())
            st.profile_enable(True)
            st.advance(zi, length, 0, rs.subcycles, rs.dzmin)
            assert (st.profile_read('exchange')[1] > 0) == (width is None)
            states.append(st.get_state())
    scale = np.max(np.abs(states[0]))
    assert np.max(np.abs(states[1] - states[0])) <= (1e-13 if precision == 'fp64' else 0.0) * scale
