'''Cartesian FP64 lines of 256 points and more: grids with few workgroups take the y passes one by one, others in one launch
with the RK stage, both against the plain FP64 stepper (1e-10), fixed and adaptive steps in two advance calls.
'''
import pytest

from conftest import rel_l2
from searay_amd import configs, uppe_kernel

pytestmark = pytest.mark.gpu


def _run(rs, precision, dzmin):
    zi, _, length = rs.plane(0)
    with rs.make_stepper(uppe_kernel.hip_stepper_factory(precision)) as st:
        st.set_field(rs.stepper_field())
        st.profile_enable(True)
        steps = [st.advance(zi, length, sub, 1, dzmin)[0] for sub in (0, 1)]
        return st.get_state(), steps, st.profile_read('exchange')[1]


@pytest.mark.parametrize('nw,nx,ny,exchange', [(17, 2, 256, False), (33, 8, 1024, False), (65, 8, 256, True),
                                               (65, 8, 1024, True), (33, 16, 512, True)])
@pytest.mark.parametrize('adaptive', [False, True])
def test_long_lines(nw, nx, ny, exchange, adaptive):
    vol = configs.cartesian_filamentation(scale=8, steps=100, length='10 cm')
    vol['wave grid'] = (nw, nx, ny, 2)
    vol['frequency band'] = (0.0, 2.0)
    vol['nonlinear band'] = (0.0, 1.4)
    rs = uppe_kernel.RunSetup(vol)
    dzmin = rs.plane(0)[2] / (20 if adaptive else 1)
    print('lines of %d: %d x %d adaptive=%s' % (ny, nw, nx, adaptive), flush=True)
    want, steps, _ = _run(rs, 'fp64-plain', dzmin)
    got, taken, launches = _run(rs, 'fp64', dzmin)
    assert taken == steps
    assert (launches > 0) == exchange
    assert rel_l2(got, want) < 1e-10
