"""Arc sums at the edges of their layout (arc_cols and ArcLayout in density_arcs.h
and kernels.h), on FP32-storage models, which take them at any size: both sides of
the changes from 8 to 4 to 2 columns per block (NU 12 and 13, 25 and 26), with the
most source texels a block loads (480 and 500 of 512 threads), 1 and 2 tiles per
wave, partial blocks in mu and mu_s, and several groups of wavelengths. Init(4)
against the FP64 oracle, by the norm of the error relative to the texture's: sums of
at most 36 terms in FP32 at each of 16 angles, 6e-8 times 600, were all to round
one way, are 3.5e-5; as independent roundings 1.5e-6; two further orders and the
march of 51 samples make it 5e-6.

The packed store of FP16-storage models, which take the arcs above 2^22 texels:
against FP32 storage at the same odd sizes, within FP16's own rounding (2^-11 of a
texel, and 2^-15 for the 21-bit density)."""
import numpy as np
import pytest

import parity
from precomputed_atmospheric_scattering_amd import configs
from test_host_rules import job, rules  # noqa: F401 (fixture)

SMALL = [(12, 15), (13, 15), (25, 15), (26, 15), (9, 9), (15, 3), (12, 3), (13, 3), (25, 3),
         (26, 3), (32, 18), (3, 15)]
LARGE = (64, 130, 67, 9)


def sizes(r, mu, mu_s, nu):
    return dict(transmittance_width=64, transmittance_height=16, scattering_r=r,
                scattering_mu=mu, scattering_mu_s=mu_s, scattering_nu=nu, irradiance_width=16,
                irradiance_height=4)


def config(z, wavelengths, half=False):
    if wavelengths == 3:
        return configs.earth(lut_sizes=z, half_precision=half)
    return configs.spectral(lut_sizes=z, half_precision=half,
                            num_precomputed_wavelengths=wavelengths)


def test_sizes_take_the_arcs(rules):  # noqa: F811
    r, mu, mu_s, nu = LARGE
    jobs = [job(nr=3, nmu=22, nmus=9, nnu=n, niter=-(-w // 3)) for n, w in SMALL]
    jobs += [job(nr=r, nmu=mu, nmus=mu_s, nnu=nu, niter=2, half=h) for h in (0, 1)]
    assert all(got[9] for got in rules(jobs))


@pytest.mark.gpu
@pytest.mark.parametrize("nu,wavelengths", SMALL)
def test_matches_oracle(nu, wavelengths):
    cfg = config(sizes(3, 22, 9, nu), wavelengths)
    ref = parity.oracle_init(cfg, 4)
    m = parity.gpu_model(cfg)
    m.init(4)
    for name in ("scattering", "irradiance"):
        want = ref[name][..., :3]
        got = np.asarray(m.lut(name), np.float64).reshape(ref[name].shape)[..., :3]
        e = np.linalg.norm(got - want) / np.linalg.norm(want)
        print(name, "%.2e" % e, flush=True)
        assert e <= 5e-6, name
    m.close()


@pytest.mark.gpu
def test_packed_store():
    luts = []
    for half in (False, True):
        m = parity.gpu_model(config(sizes(*LARGE), 6, half))
        m.init(3)
        luts.append([np.array(m.lut(n))[..., :3].reshape(-1, 3)
                     for n in ("scattering", "irradiance")])
        m.close()
    for full, half in zip(*luts):
        # Luminances are differences in single texels: by the texel's largest channel.
        scale = np.abs(full).max(axis=1, keepdims=True)
        floor = 1e-6 * scale.max()
        e = (np.abs(half - full) / np.maximum(scale, floor)).max()
        print("%.2e" % e, flush=True)
        assert e <= parity.TOL_FP16
