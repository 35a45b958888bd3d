"""The density tuner times the kernels that the shapes of a class apply to, and
density jobs that take no shape share a launch whatever shape their class has."""
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


def sizes(r, mu, mu_s, nu):
    return dict(transmittance_width=64, transmittance_height=16, scattering_r=r,
                scattering_mu=mu, scattering_mu_s=mu_s, scattering_nu=nu, irradiance_width=16,
                irradiance_height=4)


def density_ms(z):
    kw, _ = configs.model_kwargs(configs.earth(half_precision=True, lut_sizes=z))
    m = atmo.Model(pass_timing=True, **kw)
    best = 1e9
    for _ in range(5):
        m.init(4)
        best = min(best, sum(ms for p, _, ms in m.pass_timings() if p == "scattering_density"))
    m.close()
    return best


# Planes of 16 x 2 and 8 x 4 outputs: at 4 nu per thread one wave per block has 8 or
# 16 threads to work with; at 1, three times as fast (0.19 against 0.6 ms measured).
# The bound leaves room for half of that.
@pytest.mark.parametrize("mu,nu", [(16, 2), (8, 4)])
def test_tuned_shape_is_faster_for_the_models_that_use_it(mu, nu):
    z = sizes(8, mu, 16, nu)
    before = density_ms(z)
    atmo.autotune([z])
    t = atmo.get_tiles(z)
    assert t["sd_tuned"] and (t["sd_nu_per_thread"], t["sd_block_threads"]) != (4, 128)
    assert density_ms(z) < 0.65 * before


# Beyond 2^22 texels (FP32 tuning models), with order 3 by arc sums and by directions.
@pytest.mark.parametrize("z", [sizes(64, 128, 64, 9), sizes(64, 128, 32, 24)])
def test_large_classes(z):
    atmo.autotune([z])
    sd, _ = atmo.tile_candidates()
    t = atmo.get_tiles(z)
    assert t["sd_tuned"] and (t["sd_nu_per_thread"], t["sd_block_threads"]) in sd


def test_jobs_without_a_shape_share_a_launch():
    zs = [sizes(8, 32, 8, 4), sizes(8, 64, 8, 4), sizes(8, 32, 8, 6)]

    def launches():
        models = [parity.gpu_model(configs.earth(lut_sizes=z)) for z in zs]
        b = atmo.Batch(models, [3] * len(models))
        n = b.num_launches
        b.close()
        for m in models:
            m.close()
        return n

    n = launches()
    for z, (chunk, block) in zip(zs, ((1, 256), (2, 128), (4, 64))):
        atmo.set_tiles(z, chunk, block, 1, 256, ms_row_order="ray")
    assert launches() == n
