"""Scattering density of the orders >= 3 on both sides of the rule that chooses
between arc sums and directions for models of 3 wavelengths with many NU (arc_sums
in kernels.h): Init(3) with FP32 storage against FP16 storage of the same sizes,
which takes the directions on both sides, at the repository's bar for FP16 (5e-3);
and alone against a batch of both, bit for bit."""
import numpy as np
import pytest

import parity
import precomputed_atmospheric_scattering_amd as atmo
from precomputed_atmospheric_scattering_amd import configs

pytestmark = pytest.mark.gpu


def sizes(mu_s, nu):
    return dict(transmittance_width=64, transmittance_height=16, scattering_r=32,
                scattering_mu=128, scattering_mu_s=mu_s, scattering_nu=nu, irradiance_width=16,
                irradiance_height=4)


def luts(m):
    return [np.array(m.lut(n)) for n in ("scattering", "irradiance")]


def test_both_sides_of_the_limits():
    cfgs = [configs.earth(lut_sizes=sizes(*z), half_precision=h)
            for z in ((24, 19), (24, 20), (25, 19), (20, 23)) for h in (False, True)]
    models = [parity.gpu_model(c) for c in cfgs]
    alone = []
    for m in models:
        m.init(3)
        alone.append(luts(m))
    for f32, f16 in zip(alone[::2], alone[1::2]):
        for a, b in zip(f32, f16):
            assert parity.rel_err(b, a)[0] <= parity.TOL_FP16
    b = atmo.Batch(models, [3] * len(models))
    b.launch()
    atmo.synchronize()
    for m, want in zip(models, alone):
        assert all(np.array_equal(x, y) for x, y in zip(luts(m), want))
    b.close()
    for m in models:
        m.close()
