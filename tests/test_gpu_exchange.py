'''The exchange launches (the transform of one stage back to k-space and the next stage's transform out of it in one
kernel) at the edges of their tiles, against the oracle. Radial grids: fewer rows than a 16-row tile, modes that end
inside one, nonlinear bands that end inside a column tile, both tile widths, one to four row tiles per wave. Cartesian
grids: the shortest lines, lines of every first radix, the longest (8 FP32 columns per line), bands that end inside a
column tile. Every grid runs fixed, adaptive and replayed steps in two advance calls, so each stage opens, exchanges and
resumes. Tolerances as for the other parity
tests: FP64 1e-10, FP32 and BF16x3 1e-5 on the oracle's steps.
'''
import sys

import pytest

from conftest import rel_l2
from searay_amd import configs, uppe_kernel

pytestmark = pytest.mark.gpu

# (frequencies, cells, modes, share of the band that is nonlinear)
GRIDS = [(129, 8, 5, 1.0), (129, 16, 16, 0.61), (257, 32, 27, 0.43), (257, 128, 100, 1.0), (129, 256, 233, 0.7),
         (1025, 64, 50, 1.0), (2049, 32, 32, 0.5)]
# two 16-row tiles per wave on half tiles (BF16x3), four (FP64)
TALL = [(257, 512, 491, 1.0, 'bf16x3'), (1025, 512, 300, 1.0, 'fp64')]

# Cartesian: (frequencies, x cells, y cells, share of the band that is nonlinear)
LINES = [(33, 4, 2, 1.0), (33, 2, 8, 0.5), (65, 8, 16, 0.4), (33, 4, 128, 1.0), (17, 2, 1024, 0.7)]

_refs = {}


def _vol(nw, nr, nk, share):
    vol = configs.radial_o2_ionization(scale=max(1, 2048 // (nw - 1)), nr=nr, steps=3, length='0.3 mm')
    vol['wave grid'] = (nw, nr, 1, 2)
    vol['radial modes'] = nk
    band = (0.0, max(2.0, vol['frequency band'][1]))
    vol['frequency band'] = band
    vol['nonlinear band'] = (0.0, max(1.4, share * band[1]))
    return vol


def _lines_vol(nw, nx, ny, share):
    vol = configs.cartesian_filamentation(scale=8, steps=100, length='10 cm')
    vol['wave grid'] = (nw, nx, ny, 2)
    vol['frequency band'] = (0.0, 2.0)
    vol['nonlinear band'] = (0.0, 2.0 * share)
    vol['minimum step'] = 1.0
    vol['size'] = vol['size'][:2] + (vol['size'][2] * 3 / 100,)
    vol['subcycles'] = 3
    return vol


def _run(rs, factory, mode, schedule=None):
    '''The state after subcycle 0 and then 1-2, and the steps of each call.'''
    zi, _, length = rs.plane(0)
    dzmin = length if mode == 'fixed' else rs.dzmin
    with rs.make_stepper(factory) as st:
        st.set_field(rs.stepper_field())
        recs = []
        for sub0, n in ((0, 1), (1, 2)):
            sched = None if schedule is None else schedule[len(recs)]
            recs.append(st.advance(zi, length, sub0, n, dzmin, dz_schedule=sched, record_cap=64)[1])
        return st.get_state(), recs


def _check(oracle_mod, grid, precision, build=_vol):
    if grid not in _refs:
        rs = uppe_kernel.RunSetup(build(*grid))
        _refs[grid] = rs, {m: _run(rs, oracle_mod.oracle_factory, m) for m in ('fixed', 'adaptive')}
    rs, refs = _refs[grid]
    factory = uppe_kernel.hip_stepper_factory(precision)
    tol = 1e-10 if precision == 'fp64' else 1e-5
    for mode, ref in refs.items():
        print('exchange %s %s %s' % (grid, precision, mode), flush=True)
        sys.stdout.flush()
        q, recs = _run(rs, factory, mode, None if mode == 'fixed' or precision == 'fp64' else ref[1])
        assert [len(r) for r in recs] == [len(r) for r in ref[1]]
        assert rel_l2(q, ref[0]) < tol, (mode, rel_l2(q, ref[0]))


@pytest.mark.parametrize('grid', GRIDS)
@pytest.mark.parametrize('precision', ['fp64', 'fp32', 'bf16x3'])
def test_exchange_tiles(oracle_mod, grid, precision):
    _check(oracle_mod, grid, precision)


@pytest.mark.parametrize('case', TALL)
def test_exchange_row_tiles(oracle_mod, case):
    _check(oracle_mod, case[:4], case[4])


@pytest.mark.parametrize('grid', LINES)
@pytest.mark.parametrize('precision', ['fp64', 'fp32'])
def test_exchange_lines(oracle_mod, grid, precision):
    _check(oracle_mod, grid, precision, _lines_vol)
