"""Scattering density of FP16-storage models on both sides of the size from which
they take the arc sums for the orders >= 3 (fixed_sums in kernels.h): against a
model with FP32 storage, which takes them at any size, at the repository's bar
for FP16 storage (5e-3; rounding a texel to FP16 is 5e-4 of it, delta J to 3 x 21
bits 3e-5)."""
import numpy as np
import pytest

import parity
from precomputed_atmospheric_scattering_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nu", [8, 9])  # 2^22 texels, and above
def test_both_sides_of_the_limit(nu):
    sizes = dict(transmittance_width=128, transmittance_height=32, scattering_r=64,
                 scattering_mu=128, scattering_mu_s=64, scattering_nu=nu)
    luts = []
    for half in (False, True):
        m = parity.gpu_model(configs.earth(lut_sizes=sizes, half_precision=half))
        m.init(3)
        luts.append([np.array(m.lut(n)) for n in ("scattering", "single_mie_scattering")])
        m.close()
    for f32, f16 in zip(*luts):
        e, _ = parity.rel_err(f16, f32)
        assert e <= parity.TOL_FP16, e
