'''The exchange launches on the steps that test_gpu_exchange leaves out, over its grids: FP32 and BF16x3 on adaptive steps of
their own (stage 1 in two launches with the step estimate between them), FP64 on the oracle's schedule. The same step
counts and 1e-4 on the state on own steps, as for the other adaptive parity tests; FP64 1e-10 on the oracle's.
'''
import pytest

from conftest import rel_l2
from searay_amd import uppe_kernel
from test_gpu_exchange import GRIDS, LINES, _lines_vol, _refs, _run, _vol

pytestmark = pytest.mark.gpu


def _reference(oracle_mod, grid, build):
    if grid not in _refs:
        rs = uppe_kernel.RunSetup(build(*grid))
        _refs[grid] = rs, {m: _run(rs, oracle_mod.oracle_factory, m) for m in ('fixed', 'adaptive')}
    return _refs[grid][0], _refs[grid][1]['adaptive']


def _check_own_steps(oracle_mod, grid, precision, build):
    rs, ref = _reference(oracle_mod, grid, build)
    print('exchange %s %s own adaptive steps' % (grid, precision), flush=True)
    q, recs = _run(rs, uppe_kernel.hip_stepper_factory(precision), 'adaptive')
    assert [len(r) for r in recs] == [len(r) for r in ref[1]]
    assert rel_l2(q, ref[0]) < 1e-4, rel_l2(q, ref[0])


def _check_schedule(oracle_mod, grid, build):
    rs, ref = _reference(oracle_mod, grid, build)
    print('exchange %s fp64 on the oracle\'s steps' % (grid,), flush=True)
    q, recs = _run(rs, uppe_kernel.hip_stepper_factory('fp64'), 'adaptive', ref[1])
    assert [list(r) for r in recs] == [list(r) for r in ref[1]]
    assert rel_l2(q, ref[0]) < 1e-10, rel_l2(q, ref[0])


@pytest.mark.parametrize('grid', GRIDS)
@pytest.mark.parametrize('precision', ['fp32', 'bf16x3'])
def test_tiles_on_own_steps(oracle_mod, grid, precision):
    _check_own_steps(oracle_mod, grid, precision, _vol)


@pytest.mark.parametrize('grid', LINES)
def test_lines_on_own_steps(oracle_mod, grid):
    _check_own_steps(oracle_mod, grid, 'fp32', _lines_vol)


@pytest.mark.parametrize('grid', GRIDS)
def test_tiles_on_the_oracles_steps(oracle_mod, grid):
    _check_schedule(oracle_mod, grid, _vol)


@pytest.mark.parametrize('grid', LINES)
def test_lines_on_the_oracles_steps(oracle_mod, grid):
    _check_schedule(oracle_mod, grid, _lines_vol)
