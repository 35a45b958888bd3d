"""Tile shapes where they apply (sd_uses_tile in kernels.h): models with FP16
storage, whose density takes a shape at every order, and with FP32 storage above
1.25M texels, at order 2, give bit-identical LUTs for every shape, with planes and NU
that leave partial blocks and chunks. test_sizes_take_the_shapes checks on the host
that they are such models."""
import numpy as np
import pytest

import precomputed_atmospheric_scattering_amd as atmo
from precomputed_atmospheric_scattering_amd import configs
from test_host_rules import job, rules  # noqa: F401 (fixture)

NAMES = ("transmittance", "scattering", "single_mie_scattering", "irradiance")


def sizes(r, mu, mu_s, nu):
    return dict(transmittance_width=64, transmittance_height=16, scattering_r=r,
                scattering_mu=mu, scattering_mu_s=mu_s, scattering_nu=nu, irradiance_width=32,
                irradiance_height=8)


# R, MU, MU_S, NU, wavelengths, FP16, orders.
CASES = {
    "half small": (8, 64, 16, 4, 3, True, 4),
    "half odd": (5, 46, 9, 7, 3, True, 4),
    "half least": (2, 4, 2, 2, 3, True, 3),
    "half reference": (32, 128, 32, 8, 3, True, 4),
    "half spectral": (8, 64, 16, 4, 15, True, 3),
    "full above the split": (32, 128, 32, 10, 3, False, 2),
    "full odd": (31, 126, 37, 9, 3, False, 2),
    "full by directions": (32, 128, 24, 20, 3, False, 3),
    "full spectral": (16, 64, 32, 8, 15, False, 2),
}


def test_sizes_take_the_shapes(rules):  # noqa: F811
    for name, (r, mu, mu_s, nu, wavelengths, half, orders) in CASES.items():
        got = rules([job(nr=r, nmu=mu, nmus=mu_s, nnu=nu, niter=-(-wavelengths // 3),
                         half=half)])[0]
        assert got[6] == 3, name                       # order 2 has a thread per output
        assert orders == 2 or got[9] == 0, name        # and so have the orders >= 3


@pytest.fixture(autouse=True)
def clean_table():
    atmo.reset_tiles()
    yield
    atmo.reset_tiles()


def run(cfg, orders):
    kw, _ = configs.model_kwargs(cfg)
    m = atmo.Model(**kw)
    m.init(orders)
    out = {n: np.array(m.lut(n)) for n in NAMES}
    m.close()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_every_shape_gives_identical_luts(name):
    r, mu, mu_s, nu, wavelengths, half, orders = CASES[name]
    z = sizes(r, mu, mu_s, nu)
    cfg = (configs.earth(lut_sizes=z, half_precision=half) if wavelengths == 3 else
           configs.spectral(lut_sizes=z, half_precision=half,
                            num_precomputed_wavelengths=wavelengths))
    want = run(cfg, orders)
    sd, ms = atmo.tile_candidates()
    w = mu_s * nu
    d = atmo.get_tiles(z)
    dms = (d["ms_texels_per_thread"], d["ms_block_threads"])
    shapes = [(s, dms) for s in sd] + [(sd[0], t) for t in ms if w <= t[0] * t[1]]
    for (chunk, block), (tpt, mblock) in shapes:
        print("case", name, chunk, block, tpt, mblock, flush=True)
        atmo.set_tiles(z, chunk, block, tpt, mblock, ms_row_order=d["ms_row_order"])
        got = run(cfg, orders)
        for n in NAMES:
            assert np.array_equal(got[n], want[n]), (name, chunk, block, tpt, mblock, n)
