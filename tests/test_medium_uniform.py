'''The uniform-medium check of the batched and adjoint paths (host only).'''
import numpy as np
import pytest

from searay_amd import configs, uppe_kernel, volume


class TestUniformMedium:
    '''RunSetup.medium_is_uniform: the evaluation of all planes at once agrees with the planes one by one.'''

    @pytest.mark.parametrize('density, uniform', [
        (lambda x, y, z, r2: np.ones(r2.shape), True),
        (lambda x, y, z, r2: np.exp(-r2 / 1e8), True),
        (lambda x, y, z, r2: 1.0, True),
        (lambda x, y, z, r2: np.ones(r2.shape) + 1e-9 * z, False),
        (lambda x, y, z, r2: np.where(np.abs(z) < 5000.0, 0.5, 1.0) * np.ones(r2.shape), False),
        (lambda x, y, z, r2: np.where(z > 0, np.nan, 1.0) * np.ones(r2.shape), False),
    ])
    def test_against_planes_one_by_one(self, density, uniform, monkeypatch):
        vol = configs.radial_o2_ionization(scale=8, steps=12, length='1 cm')
        vol['density lambda'] = density
        rs = uppe_kernel.RunSetup(vol)
        assert rs.medium_is_uniform(0) is uniform
        monkeypatch.setattr(uppe_kernel.RunSetup, '_same_in_one_evaluation', lambda self, zs, d0: False)
        assert rs.medium_is_uniform(0) is uniform

    def test_other_volumes_are_asked_plane_by_plane(self):
        class Box(volume.AnalyticBox):
            def GetRelDensity(self, xp):
                return np.full(xp.shape[:-1], 1.0 + (xp[0, 0, 3] > 0))
        vol = configs.radial_o2_ionization(scale=8, steps=12, length='1 cm')
        vol['object'] = Box('air')
        vol['object'].Initialize(vol)
        assert uppe_kernel.RunSetup(vol).medium_is_uniform(0) is False
