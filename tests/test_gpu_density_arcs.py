"""Scattering density of orders >= 3 (arc sums): Init(4) against the FP64
oracle at the edges of the kernel's layout. The bars are the repository's
(1e-3 FP32, 5e-3 FP16): an azimuth, a term or a texel left out or counted
twice changes a density by percents."""
import pytest

import parity
from precomputed_atmospheric_scattering_amd import configs

pytestmark = pytest.mark.gpu

# NU: smallest, one and two tiles per wave (4, 5), 8 and 4 columns per block
# (14, 15), whole and partial tiles, largest. MU and MU_S leave partial blocks.
# Wavelengths: 1 to 4 groups of 4, and a second group of iterations (18).
CASES = [(2, 3, False), (4, 3, False), (5, 6, False), (8, 15, False), (9, 9, True),
         (14, 12, False), (15, 3, True), (16, 18, False), (32, 3, False)]


def sizes(nnu, **kw):
    return dict(dict(transmittance_width=64, transmittance_height=16, scattering_r=3,
                     scattering_mu=22, scattering_mu_s=9, scattering_nu=nnu,
                     irradiance_width=16, irradiance_height=4), **kw)


@pytest.mark.parametrize("nnu,wavelengths,half", CASES)
def test_orders_match_oracle(nnu, wavelengths, half):
    if wavelengths == 3:
        cfg = configs.earth(lut_sizes=sizes(nnu), half_precision=half)
    else:
        cfg = configs.spectral(lut_sizes=sizes(nnu), half_precision=half,
                               num_precomputed_wavelengths=wavelengths)
    errs = parity.compare_init(cfg, 4)
    assert all(e <= (parity.TOL_FP16 if half else parity.TOL_FP32) for e in errs.values()), errs


def test_more_terms_than_held():
    # A thick atmosphere over a small planet and a fine irradiance LUT: the
    # ground irradiance has over 100 breakpoints at some angles.
    cfg = configs.earth(lut_sizes=sizes(6, scattering_r=4, irradiance_width=500))
    cfg.update(bottom_radius=1000e3, top_radius=1300e3, ground_albedo=[0.9] * 3)
    errs = parity.compare_init(cfg, 4)
    assert all(e <= parity.TOL_FP32 for e in errs.values()), errs
