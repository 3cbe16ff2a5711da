'''The uniform-medium check of the batched and adjoint paths against the density asked plane by plane, for lambdas that
read their plane's z as one number, reduce over their arguments or write to them (host only). In each the interval's
ends are alike, so only its interior tells.
'''
import numpy as np
import pytest

from searay_amd import configs, uppe_kernel, volume


def _setup(density):
    vol = configs.radial_o2_ionization(scale=8, steps=16, length='1 cm')
    vol['density lambda'] = density
    return uppe_kernel.RunSetup(vol)


def _plane_by_plane(density):
    rs = _setup(density)
    zi, _, L = rs.plane(0)
    d0 = rs.mat.density(zi + 0.5 * L)
    return all(np.array_equal(rs.mat.density(zi + sub * L + 0.5 * L), d0) for sub in range(rs.subcycles))


S = _setup(lambda x, y, z, r2: np.ones(r2.shape)).size[3]


def _shifts_its_points(x, y, z, r2):
    x += 1.0 * (np.abs(z) < S / 4)
    return np.ones(r2.shape) + (x[0, 0] > 4 * S)


def _writes_r2(x, y, z, r2):
    r2 *= 1e-9
    return np.exp(-r2, out=r2)


def _reads_where_r2_was_written(x, y, z, r2):
    r2 += np.abs(z[0, 0])
    return (r2 >= 0) * (1.0 if np.abs(z[0, 0]) > S / 4 else 0.5)


VARYING = [
    lambda x, y, z, r2: np.ones(r2.shape) * (1.0 if abs(z[0, 0]) < S / 4 else 0.5),
    lambda x, y, z, r2: np.ones(r2.shape) * np.exp(-(z[0, 0] / S) ** 2),
    lambda x, y, z, r2: np.ones_like(r2) * (0.5 if abs(z.flat[0]) > S / 4 else 1.0),
    lambda x, y, z, r2: np.ones_like(r2) * (0.5 if np.abs(z).max() > S / 4 else 1.0),
    lambda x, y, z, r2: np.ones_like(r2) if np.all(np.abs(z) < S / 4) else 0.5 * np.ones_like(r2),
    lambda x, y, z, r2: np.interp(z[0, 0], [-S, -S / 4, 0, S / 4, S], [1.0, 1.0, 0.5, 1.0, 1.0]) * np.ones(r2.shape),
    lambda x, y, z, r2: np.full(r2.shape, 1.0 + (z.min() > -S / 4) * (z.max() < S / 4)),
    lambda x, y, z, r2: 0.5 if abs(z[0, 0]) < S / 4 else np.ones(r2.shape),
    _reads_where_r2_was_written,
]
UNIFORM = [
    lambda x, y, z, r2: np.ones(r2.shape) * (1.0 if abs(z[0, 0]) < 4 * S else 0.5),
    lambda x, y, z, r2: np.exp(-r2 / np.max(r2)),
    lambda x, y, z, r2: np.full(r2.shape, z.size / z.size),
    _writes_r2,
]


@pytest.mark.parametrize('density', VARYING)
def test_interior_that_differs_is_refused(density):
    assert not _plane_by_plane(density)
    assert _setup(density).medium_is_uniform(0) is False


@pytest.mark.parametrize('density', UNIFORM)
def test_uniform_media_are_taken(density):
    assert _plane_by_plane(density)
    assert _setup(density).medium_is_uniform(0) is True


def test_a_lambda_that_moves_its_points():
    assert _setup(_shifts_its_points).medium_is_uniform(0) is _plane_by_plane(_shifts_its_points)


def test_a_lambda_that_asks_for_one_plane():
    def density(x, y, z, r2):
        assert x.shape == y.shape == z.shape == r2.shape and r2.ndim == 2
        assert z.flags.writeable and r2.flags.writeable and np.ptp(z) == 0.0
        return np.ones(r2.shape)
    assert _setup(density).medium_is_uniform(0) is True


def test_a_density_set_on_the_volume_is_asked():
    rs = _setup(lambda x, y, z, r2: np.ones(r2.shape))
    assert isinstance(rs.mat.vol, volume.AnalyticBox)
    rs.mat.vol.GetRelDensity = lambda xp: np.full(xp.shape[:-1], 1.0 if abs(xp[0, 0, 3]) < S / 4 else 0.5)
    assert rs.medium_is_uniform(0) is False
