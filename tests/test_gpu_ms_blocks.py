"""Multiple scattering: the blocks' ways of dealing out a row give the same bits.
FP16-storage models whose launches have 2048 blocks or fewer (a texel per load or
two, ms_pairs in kernels.h), against the tile of two texels per thread, which
always loads two; rows alone in a block, of few blocks (ms_spread) and more,
against a tile of another width; odd rows, and rows that fill a block."""
import numpy as np
import pytest

import parity
import precomputed_atmospheric_scattering_amd as atmo
from precomputed_atmospheric_scattering_amd import configs

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def clean_table():
    atmo.reset_tiles()
    yield
    atmo.reset_tiles()


def luts(cfg, sizes, tpt, block):
    atmo.set_tiles(sizes, 4, 128, tpt, block)
    m = parity.gpu_model(cfg)
    m.init(3)
    out = [np.array(m.lut(n)) for n in ("scattering", "irradiance")]
    m.close()
    return out


def sizes(r, mu, mu_s, nu):
    return dict(transmittance_width=64, transmittance_height=16, scattering_r=r,
                scattering_mu=mu, scattering_mu_s=mu_s, scattering_nu=nu, irradiance_width=16,
                irradiance_height=4)


# R, MU, MU_S, NU, wavelengths: 2048 blocks and 2046 or 2040 of rows of 256, 129
# and 27 (7 rows a block), 5 iterations; few blocks.
@pytest.mark.parametrize("r,mu,mu_s,nu,wavelengths", [
    (32, 64, 32, 8, 3), (33, 62, 32, 8, 3), (32, 64, 43, 3, 3), (33, 62, 43, 3, 3),
    (41, 70, 9, 3, 15), (40, 70, 9, 3, 15), (3, 10, 9, 3, 3), (2, 4, 2, 2, 15)])
def test_texel_loads(r, mu, mu_s, nu, wavelengths):
    z = sizes(r, mu, mu_s, nu)
    cfg = (configs.earth(half_precision=True, lut_sizes=z) if wavelengths == 3 else
           configs.spectral(half_precision=True, lut_sizes=z,
                            num_precomputed_wavelengths=wavelengths))
    want = luts(cfg, z, 2, 256)
    got = luts(cfg, z, 1, 256)
    assert all(np.array_equal(a, b) for a, b in zip(got, want))


# Rows of 257, 300, 511 and 512 alone in blocks of 256 and of 512 threads.
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("r", [3, 26])  # 30 and 260 rows
@pytest.mark.parametrize("mu_s,nu", [(257, 2), (100, 3), (73, 7), (64, 8), (171, 3)])
def test_row_per_block(mu_s, nu, r, half):
    z = sizes(r, 10, mu_s, nu)
    cfg = configs.earth(half_precision=half, lut_sizes=z)
    w = mu_s * nu
    if w > 512:
        errs = parity.compare_init(cfg, 2)
        assert all(e <= (parity.TOL_FP16 if half else parity.TOL_FP32) for e in errs.values())
        return
    want = luts(cfg, z, 2, 512)
    got = luts(cfg, z, 2, 256)
    assert all(np.array_equal(a, b) for a, b in zip(got, want))
