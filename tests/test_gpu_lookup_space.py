"""GetSkyRadiance where whole waves of rays miss the atmosphere, others partly,
and the last wave is not full: with and without a lookup copy the same bits, and
no radiance and full transmittance for the rays that miss it. Each of the three
kernels (combined; separate with a copy; without) is compared with the oracle's
definition of those rays only; the rest is in test_gpu_queries.py and
test_gpu_lookup_lines.py."""
import numpy as np
import pytest

import precomputed_atmospheric_scattering_amd as atmo
from precomputed_atmospheric_scattering_amd import configs

pytestmark = pytest.mark.gpu

SIZES = dict(transmittance_width=64, transmittance_height=16, scattering_r=8, scattering_mu=32,
             scattering_mu_s=9, scattering_nu=7, irradiance_width=16, irradiance_height=4)


def rays(n, rb, rt, mix):
    q = {k: np.array(v) for k, v in configs.sky_queries(9, n, rb, rt).items()}
    r = np.linalg.norm(q["camera"], axis=1)
    q["camera"] *= (np.minimum(r, rt - 1.0) / r)[:, None].astype(np.float32)
    i = np.arange(n)
    miss = {"all": i >= 0, "waves": i // 64 % 2 == 0, "lanes": i % 3 == 0, "last": i >= n - 1,
            "but one": i != 70 % n}[mix]
    q["camera"][miss] = np.float32([0.0, 0.0, 1.5 * rt])
    q["view_ray"][miss] = np.float32([0.6, 0.0, 0.8])
    return q, miss


@pytest.mark.parametrize("mix", ["all", "waves", "lanes", "last", "but one"])
@pytest.mark.parametrize("n", [1, 64, 130, 1000])
@pytest.mark.parametrize("half", [False, True])
def test_rays_in_space(half, n, mix):
    kw, _ = configs.model_kwargs(configs.earth(half_precision=half, lut_sizes=SIZES))
    rb, rt = kw["bottom_radius"] / 1000.0, kw["top_radius"] / 1000.0
    q, miss = rays(n, rb, rt, mix)
    out = []
    for combined, copy in ((False, True), (False, False), (True, False)):
        kw["combine_scattering_textures"] = combined
        m = atmo.Model(interleaved_lookups=copy, **kw)
        m.init(2)
        for shadow in (0.0, 1.5):
            rad, tr = m.sky_radiance(q["camera"], q["view_ray"], np.full(n, shadow, np.float32),
                                     q["sun_direction"])
            assert np.isfinite(rad).all() and (rad[miss] == 0).all() and (tr[miss] == 1).all()
            assert (tr[~miss] < 1).all()
            out.append((rad, tr))
        m.close()
    for a, b in zip(out[:2], out[2:4]):
        assert all(np.array_equal(x, y) for x, y in zip(a, b))
