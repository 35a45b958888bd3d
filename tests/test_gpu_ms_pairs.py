"""Multiple scattering of FP16-storage models, whose blocks read pairs of texels
of packed rows (MU_S x NU texels), against the FP64 oracle at the repository's bar
for FP16 storage: odd rows (the last pair overlaps), the shortest, several rows
per block, a partial last block, and each tile shape. A texel left out or taken
from its neighbour is off by percents."""
import pytest

import parity
from precomputed_atmospheric_scattering_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mu_s,nu", [(2, 2), (9, 3), (15, 17), (16, 16), (33, 9), (43, 6),
                                     (73, 7), (67, 11), (64, 16)])
def test_rows(mu_s, nu):
    cfg = configs.earth(half_precision=True, lut_sizes=dict(
        transmittance_width=64, transmittance_height=16, scattering_r=3, scattering_mu=10,
        scattering_mu_s=mu_s, scattering_nu=nu, irradiance_width=16, irradiance_height=4))
    errs = parity.compare_init(cfg, 2)
    assert all(e <= parity.TOL_FP16 for e in errs.values()), errs


@pytest.mark.parametrize("tpt,block", [(1, 256), (2, 256), (2, 512)])
def test_tiles_of_odd_rows(tpt, block):
    import precomputed_atmospheric_scattering_amd as atmo
    sizes = dict(transmittance_width=64, transmittance_height=16, scattering_r=5,
                 scattering_mu=10, scattering_mu_s=9, scattering_nu=3, irradiance_width=16,
                 irradiance_height=4)  # rows of 27
    try:
        atmo.set_tiles(sizes, 4, 128, tpt, block)
        errs = parity.compare_init(configs.earth(half_precision=True, lut_sizes=sizes), 2)
    finally:
        atmo.reset_tiles()
    assert all(e <= parity.TOL_FP16 for e in errs.values()), errs
