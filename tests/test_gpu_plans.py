'''Which kernels a radial step takes: exchanges up to 256 cells, separate contractions above and where one tile more than
the CUs would take a second round; there the exchange measured slower.
'''
import numpy as np
import pytest

from searay_amd import batch, configs, uppe_kernel

pytestmark = pytest.mark.gpu


def _vol(nw, nr, share=1.0):
    vol = configs.batched_radial(n=1, steps=200)[0][0]
    vol['wave grid'] = (nw, nr, 1, 2)
    vol['radial modes'] = nr
    vol['nonlinear band'] = (0.0, share * vol['frequency band'][1])
    return vol


def _launches(vol, precision):
    rs = uppe_kernel.RunSetup(vol)
    zi, _, length = rs.plane(0)
    with rs.make_stepper(uppe_kernel.hip_stepper_factory(precision)) as st:
        st.set_field(rs.stepper_field())
        st.profile_enable(True)
        st.advance(zi, length, 0, rs.subcycles, rs.dzmin, max_steps=2)
        return {c: st.profile_read(c)[1] for c in ('hankel', 'hankel_r2k', 'exchange')}


@pytest.mark.parametrize('nw,precision', [(129, 'bf16x3'), (513, 'bf16x3'), (513, 'fp32'), (1025, 'fp64'),
                                          (2049, 'fp64')])
def test_tall_grids_take_separate_contractions(nw, precision):
    print('plan of %d x 512 %s' % (nw, precision), flush=True)
    assert _launches(_vol(nw, 512), precision) == {'hankel': 8, 'hankel_r2k': 8, 'exchange': 0}


@pytest.mark.parametrize('nr', [8, 128, 256])
@pytest.mark.parametrize('precision', ['fp64', 'fp32', 'bf16x3'])
def test_other_grids_take_exchanges(nr, precision):
    print('plan of 257 x %d %s' % (nr, precision), flush=True)
    assert _launches(_vol(257, nr), precision) == {'hankel': 0, 'hankel_r2k': 0, 'exchange': 9}


@pytest.mark.parametrize('precision', ['fp64', 'fp32', 'bf16x3'])
@pytest.mark.parametrize('columns,exchange', [(2049, False), (2048, True)])
def test_one_tile_more_than_the_cus(precision, columns, exchange):
    print('plan of 2049 x 256 %s, %d nonlinear columns' % (precision, columns), flush=True)
    vol = _vol(2049, 256, (columns + 0.3) / 2049)
    rs = uppe_kernel.RunSetup(vol)
    assert rs.nl_filter[columns - 1] == 1.0 and not rs.nl_filter[columns:].any()
    n = _launches(vol, precision)
    assert (n['exchange'] > 0) == exchange and (n['hankel'] > 0) != exchange


@pytest.mark.parametrize('nr', [64, 512])
@pytest.mark.parametrize('precision', ['fp64', 'fp32', 'bf16x3'])
def test_tuned_handles_time_what_they_launch(nr, precision, monkeypatch):
    '''SEARAY_UPPE_TUNE=1 times candidates of the launches that the steps take, and of no others, and changes no
    result.'''
    print('tuned handle 257 x %d %s' % (nr, precision), flush=True)
    vol = _vol(257, nr)
    rs = uppe_kernel.RunSetup(vol)
    zi, _, length = rs.plane(0)
    states, counts = [], []
    for tune in ('0', '1'):
        monkeypatch.setenv('SEARAY_UPPE_TUNE', tune)
        with rs.make_stepper(uppe_kernel.hip_stepper_factory(precision)) as st:
            st.set_field(rs.stepper_field())
            st.profile_enable(True)
            st.advance(zi, length, 0, rs.subcycles, rs.dzmin, max_steps=2)
            counts.append({c: st.profile_read(c)[1] for c in ('hankel', 'hankel_r2k', 'exchange')})
            states.append(st.get_state())
    taken = {c for c, n in counts[0].items() if n > 0}
    assert {c for c, n in counts[1].items() if n > counts[0][c]} == taken
    assert all(counts[1][c] == 0 for c in counts[1] if c not in taken)
    assert np.array_equal(states[0], states[1])


@pytest.mark.parametrize('nr,members,precision,autotune,exchange', [
    (128, 16, 'bf16x3', True, False), (128, 16, 'bf16x3', False, True), (128, 12, 'bf16x3', True, True),
    (64, 32, 'bf16x3', True, True), (256, 16, 'fp32', True, False), (256, 8, 'fp32', True, True),
    (256, 16, 'fp64', True, True)])
def test_large_tuned_batches_take_separate_contractions(nr, members, precision, autotune, exchange):
    print('plan of %d x 513 x %d %s autotune=%s' % (members, nr, precision, autotune), flush=True)
    vols = configs.batched_radial(n=members, scale=2, steps=200)[0]
    for vol in vols:
        vol['wave grid'] = (513, nr, 1, 2)
        vol['radial modes'] = nr
    with batch.Batch(vols, precision=precision, autotune=autotune) as b:
        b.set_fields()
        b.advance(max_steps=1)  # times the plans
        b.set_fields()
        b.members[0].profile_enable(True)
        b.advance(max_steps=2)
        assert b.plan(0)['run_length'] == members
        n = {c: b.members[0].profile_read(c)[1] for c in ('hankel', 'hankel_r2k', 'exchange')}
        q = b.members[members - 1].get_state()
    assert (n['exchange'] > 0) == exchange and (n['hankel_r2k'] > 0) != exchange
    rs = uppe_kernel.RunSetup(vols[-1])
    zi, _, length = rs.plane(0)
    with rs.make_stepper(uppe_kernel.hip_stepper_factory(precision)) as st:
        st.set_field(rs.stepper_field())
        st.advance(zi, length, 0, rs.subcycles, rs.dzmin, max_steps=2)
        want = st.get_state()
    assert np.linalg.norm(q - want) < (1e-12 if precision == 'fp64' else 1e-5) * np.linalg.norm(want)
