'''Contractions with two 16-row tiles per wave (column tiles that fill the CUs, more than 256 rows): the last column tile
wider than the others, all alike, contractions on either side of 512 rows, modes that end inside a row tile, against the
plain FP64 stepper. FP64 1e-10, FP32 and BF16x3 1e-5 on its steps.
'''
import pytest

from conftest import rel_l2
from searay_amd import configs, uppe_kernel

pytestmark = pytest.mark.gpu

_refs = {}


def _run(rs, precision, schedule=None):
    zi, _, length = rs.plane(0)
    with rs.make_stepper(uppe_kernel.hip_stepper_factory(precision)) as st:
        st.set_field(rs.stepper_field())
        _, rec = st.advance(zi, length, 0, rs.subcycles, rs.dzmin, dz_schedule=schedule, record_cap=16, max_steps=3)
        return st.get_state(), rec


@pytest.mark.parametrize('nw,nr,nk', [(2049, 512, 391), (4097, 512, 512), (2049, 1024, 700)])
@pytest.mark.parametrize('precision', ['fp64', 'fp32', 'bf16x3'])
def test_two_row_tiles(nw, nr, nk, precision):
    if (nw, nr, nk) not in _refs:
        vol = configs.radial_o2_ionization(nr=nr, steps=3, length='0.3 mm', power=1.0)
        vol['wave grid'] = (nw, nr, 1, 2)
        vol['radial modes'] = nk
        rs = uppe_kernel.RunSetup(vol)
        _refs.clear()
        _refs[nw, nr, nk] = rs, _run(rs, 'fp64-plain')
    rs, (want, schedule) = _refs[nw, nr, nk]
    print('two row tiles per wave: %d x %d, %d modes, %s' % (nw, nr, nk, precision), flush=True)
    got, _ = _run(rs, precision, schedule)
    assert rel_l2(got, want) < (1e-10 if precision == 'fp64' else 1e-5), rel_l2(got, want)
