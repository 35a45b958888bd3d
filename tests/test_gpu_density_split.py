"""Scattering density of order 2 on grids whose outputs take several threads
each (kSdSplit in kernels.h), against the FP64 oracle, at both sides of each
size limit and with partial blocks. The bar is the repository's 1e-3 (a zenith
angle left out or counted twice changes a density by percents); FP32 sums of 2
to 16 parts round no further than one sum of 16."""
import pytest

import parity
from precomputed_atmospheric_scattering_amd import configs

pytestmark = pytest.mark.gpu

# R, MU, MU_S, NU: smallest; 16 parts up to 65536 texels (partial blocks, then
# exactly the limit); 8 parts above, with a partial chunk of NU, and up to
# 262144; 4 parts above.
CASES = [(2, 4, 2, 2), (3, 22, 5, 3), (8, 64, 32, 4), (9, 46, 31, 6), (8, 128, 32, 8),
         (9, 128, 33, 7)]


@pytest.mark.parametrize("r,mu,mu_s,nu", CASES)
def test_order_two_matches_oracle(r, mu, mu_s, nu):
    cfg = configs.earth(lut_sizes=dict(
        transmittance_width=64, transmittance_height=16, scattering_r=r, scattering_mu=mu,
        scattering_mu_s=mu_s, scattering_nu=nu, irradiance_width=16, irradiance_height=4))
    errs = parity.compare_init(cfg, 2)
    assert all(e <= parity.TOL_FP32 for e in errs.values()), errs


def test_iterations_count():
    # 5 iterations of 16384 texels take the 8 parts that one would not.
    cfg = configs.spectral(lut_sizes=dict(
        transmittance_width=64, transmittance_height=16, scattering_r=4, scattering_mu=64,
        scattering_mu_s=16, scattering_nu=4, irradiance_width=16, irradiance_height=4))
    errs = parity.compare_init(cfg, 2)
    assert all(e <= parity.TOL_FP32 for e in errs.values()), errs
