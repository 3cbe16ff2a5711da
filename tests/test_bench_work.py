'''The benchmark's algorithmic bytes and flops of an exchange launch, against a list of what the launches of one step read,
write and multiply (host only).
'''
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402
from searay_amd import configs, uppe_kernel  # noqa: E402


def _launches(f1, rest, nr, nk, c, adaptive):
    '''(bytes, products) of every exchange launch of one step inside a subcycle; c: bytes of a complex value.'''
    tables = 8 + c  # phase and kz
    fwd, back = f1 * nr * c, f1 * nr * c  # J_r in, E_r out
    linear = rest * (nk * (tables + c) + nr * c)
    out = []
    for stage in (1, 2, 3, 4):
        points = f1 * nk * (tables + c + (c if stage < 4 else 4 * c))  # q in, the slope out or three in and q out
        moved = stage in (1, 3)
        if adaptive and stage == 1:
            out.append((fwd + points, f1))
            out.append((f1 * nk * (tables + 2 * c) + back + linear, f1 + rest))
        else:
            out.append((fwd + points + back + (linear if moved else 0), 2 * f1 + (rest if moved else 0)))
    return out


@pytest.mark.parametrize('adaptive', [False, True])
@pytest.mark.parametrize('precision,el,products', [('fp64', 8, 1), ('fp32', 4, 1), ('bf16x3', 4, 4)])
@pytest.mark.parametrize('share', [0.5, 1.0])
def test_exchange_work(share, precision, el, products, adaptive):
    vol = configs.radial_o2_ionization(scale=16, nr=16, steps=2, length='0.2 mm')
    vol['radial modes'] = 11
    vol['nonlinear band'] = (0.0, share * vol['frequency band'][1])
    rs = uppe_kernel.RunSetup(vol)
    f1 = bench.nl_columns(rs)
    steps = _launches(f1, rs.N[0] - f1, 16, 11, 2 * el, adaptive)
    nbytes, flops = bench.kernel_work(rs, 'exchange', el, precision, adaptive)
    assert nbytes == pytest.approx(sum(b for b, _ in steps) / len(steps), rel=1e-12)
    assert flops == pytest.approx(sum(n for _, n in steps) * 4 * 11 * 16 * products / len(steps), rel=1e-12)


def test_roofline_tells_adaptive_steps():
    rs = uppe_kernel.RunSetup(configs.radial_o2_ionization(scale=16, nr=16, steps=2, length='0.2 mm'))
    for launches, sources, adaptive in ((41, 40, False), (51, 40, True), (5, 4, False), (6, 4, True)):
        classes = dict(exchange=(1.0, launches), source=(0.5, sources))
        r = bench.roofline_of(rs, 'fp32', classes, 0.1)
        assert r['bytes_per_launch'] == bench.kernel_work(rs, 'exchange', 4, 'fp32', adaptive)[0]
