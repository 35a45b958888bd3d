"""Single scattering on both sides of the rule that chooses its blocks (SsTiling
in kernels.h): Init(1) against the FP64 oracle.

3 wavelengths, each texel: 51 samples of about 6 FP32 roundings (6e-8), were they
all to add up, are 2e-5; the FP32 column coordinate of a transmittance above 1e-6
(an optical depth below 14, which changes by at most about 100 over the LUT's
width) is off by at most 3e-7, 3e-5 of the transmittance; twice both is 1e-4.

More wavelengths: sums in FP64 of products of two FP32 transmittances, 2e-7 of
each wavelength's radiance with the LUT's own rounding. A luminance is a sum over
the wavelengths with weights of both signs, which cancel in single texels, so the
bound is on the error's norm relative to the texture's: with weights whose
magnitudes add up to less than 5 times their sum, 1e-6."""
import numpy as np
import pytest

import parity
from precomputed_atmospheric_scattering_amd import configs

pytestmark = pytest.mark.gpu

# TW, R, MU, MU_S, NU, wavelengths.
CASES = [
    # Rows of 190 and 192 texels, gathered; TW of 4 columns a texel and beyond.
    (64, 16, 32, 95, 2, 3), (64, 16, 32, 48, 4, 3),
    (768, 16, 32, 48, 4, 3), (769, 16, 32, 48, 4, 3), (768, 16, 32, 48, 4, 15),
    # Wide transmittance over short and long rows.
    (4096, 4, 16, 13, 5, 3), (4096, 4, 16, 13, 5, 15), (4096, 2, 8, 64, 16, 15),
    # Few blocks: 510, 512; with 3 iterations staged from 512 on.
    (64, 15, 34, 32, 8, 3), (64, 16, 32, 32, 8, 3), (64, 15, 34, 32, 8, 9),
    (64, 16, 32, 32, 8, 9),
    # 768 blocks gather, 780 stage; rows of 160 on; 2 columns a texel and beyond.
    (64, 16, 48, 32, 8, 3), (64, 15, 52, 32, 8, 3), (64, 15, 52, 40, 4, 3),
    (384, 15, 52, 48, 4, 3), (385, 15, 52, 48, 4, 3),
    # Rows of 513..768: 256 threads to TW 512, then 512.
    (512, 8, 34, 57, 9, 3), (513, 8, 34, 57, 9, 3), (512, 6, 30, 64, 12, 15),
    (513, 6, 30, 64, 12, 15),
    # Blocks of 512: 2 columns a thread, 4 with 2 iterations, the LDS of more.
    (1024, 10, 40, 33, 8, 3), (1025, 10, 40, 33, 8, 3), (2048, 10, 40, 33, 8, 6),
    (2048, 10, 40, 33, 8, 9),
    # Gathered by 256 threads, iterations alone and shared (768 blocks).
    (64, 12, 64, 13, 5, 15), (64, 12, 62, 13, 5, 15), (512, 12, 64, 13, 5, 15),
    (64, 12, 64, 13, 5, 6), (64, 12, 64, 13, 5, 18), (96, 24, 32, 8, 4, 9),
]


@pytest.mark.parametrize("tw,r,mu,mu_s,nu,wavelengths", CASES)
def test_matches_oracle(tw, r, mu, mu_s, nu, wavelengths):
    z = dict(transmittance_width=tw, transmittance_height=16, scattering_r=r, scattering_mu=mu,
             scattering_mu_s=mu_s, scattering_nu=nu, irradiance_width=16, irradiance_height=4)
    if wavelengths == 3:
        cfg = configs.earth(lut_sizes=z)
        errs = parity.compare_init(cfg, 1)
        assert all(e <= 1e-4 for e in errs.values()), errs
        return
    cfg = configs.spectral(lut_sizes=z, num_precomputed_wavelengths=wavelengths)
    ref = parity.oracle_init(cfg, 1)
    m = parity.gpu_model(cfg)
    m.init(1)
    for name in ("scattering", "single_mie_scattering"):
        want = ref[name][..., :3]
        got = np.asarray(m.lut(name), np.float64).reshape(ref[name].shape)[..., :3]
        e = np.linalg.norm(got - want) / np.linalg.norm(want)
        print(name, "%.2e" % e, flush=True)
        assert e <= 1e-6, name
    m.close()
