"""Lookups whose waves read the lookup copy's lines together (lookup_lines in
query.hip): bit-identical to the same rays of a model without a copy, where each
lane reads its own texels, at the sizes and mixes where lanes could get
another's line: batches that leave a wave or block partly empty, rays of one
place (lanes load their own lines), of two places in turn and of half a wave, and
rays that miss the atmosphere among others."""
import numpy as np
import pytest

import precomputed_atmospheric_scattering_amd as atmo
from precomputed_atmospheric_scattering_amd import configs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[False, True])
def models(request):
    cfg = configs.earth(half_precision=request.param, lut_sizes=dict(
        transmittance_width=64, transmittance_height=16, scattering_r=8, scattering_mu=32,
        scattering_mu_s=9, scattering_nu=7, irradiance_width=16, irradiance_height=4))
    kw, _ = configs.model_kwargs(cfg)
    a, b = atmo.Model(**kw), atmo.Model(interleaved_lookups=False, **kw)
    a.init(2)
    b.init(2)
    yield a, b, kw["bottom_radius"] / 1000.0, kw["top_radius"] / 1000.0
    a.close()
    b.close()


def rays(n, rb, rt, mix):
    q = configs.sky_queries(5, n, rb, rt)
    q = {k: np.array(v) for k, v in q.items()}
    i = np.arange(n)
    src = {"scattered": i, "one": 0 * i, "pairs": i // 2, "turns": i % 2,
           "half wave": np.where(i % 64 < 32, 0, i), "space": i}[mix]
    q = {k: v[src] for k, v in q.items()}
    if mix == "space":
        q["camera"][::3] = np.float32([0.0, 0.0, 2.0 * rt])
        q["view_ray"][::3] = np.float32([0.0, 0.0, 1.0])
    shadow = np.where(i % 5 == 0, 1.5, 0.0).astype(np.float32)
    return q, shadow


@pytest.mark.parametrize("mix", ["scattered", "one", "pairs", "turns", "half wave", "space"])
@pytest.mark.parametrize("n", [1, 63, 65, 257, 1000])
def test_equal_without_copy(models, n, mix):
    a, b, rb, rt = models
    q, shadow = rays(n, rb, rt, mix)

    def lookups(m):
        return (m.sky_radiance(q["camera"], q["view_ray"], shadow, q["sun_direction"]) +
                m.sky_radiance_to_point(q["camera"], q["point"], shadow, q["sun_direction"]))

    for x, y in zip(lookups(a), lookups(b)):
        assert np.isfinite(x).all() and np.array_equal(x, y)
