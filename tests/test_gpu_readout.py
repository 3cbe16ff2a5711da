'''Setting a field and reading it back: the transforms outside the steps at the edges of their tiles (modes that end
inside a 16-row and a 64-row tile, contractions that end inside a chunk, both tile heights), against the same two products
in numpy, and the field alone against the field read with its diagnostics. FP64 1e-13, FP32 1e-5 (sums of at most 512
terms).
'''
import numpy as np
import pytest

from conftest import rel_l2
from searay_amd import configs, uppe_kernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nw,nr,nk', [(65, 4, 3), (65, 16, 13), (129, 128, 71), (257, 64, 64), (2049, 512, 257)])
@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
def test_set_and_read(nw, nr, nk, precision):
    vol = configs.radial_kerr_air(scale=max(1, 512 // (nw - 1)), steps=2)
    vol['wave grid'] = (nw, nr, 1, 2)
    vol['radial modes'] = nk
    print('set and read %d x %d, %d modes, %s' % (nw, nr, nk, precision), flush=True)
    rs = uppe_kernel.RunSetup(vol)
    tool = rs.field_tool.GetTransverseTool()
    lam = np.asarray(tool.Lambda).reshape(-1)
    h = np.asarray(tool.H).reshape(tool.Nk, nr)
    rng = np.random.default_rng(3)
    a = rng.standard_normal((nw, nr, 1)) + 1j * rng.standard_normal((nw, nr, 1))
    modes = np.einsum('kj,fj->fk', h * lam[None, :] / lam[:tool.Nk, None], a[:, :, 0])
    want = np.einsum('jk,fk->fj', h.T * lam[None, :tool.Nk] / lam[:, None], modes)
    tol = 1e-13 if precision == 'fp64' else 1e-5
    with rs.make_stepper(uppe_kernel.hip_stepper_factory(precision)) as st:
        st.set_field(a)
        assert rel_l2(st.get_state()[:, :tool.Nk, 0], modes) < tol
        alone = st.finish(0.0, want_diagnostics=False)[0]
        assert rel_l2(alone[:, :, 0], want) < tol
        st.set_field(a)
        assert np.array_equal(st.finish(0.0)[0], alone)
