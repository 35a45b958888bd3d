"""Batches whose models take different kernels in one pass level equal each model
precomputed alone, bit for bit: iterations served with the first of their group
(SsTiling::nit 0, blocks_density_arcs 0) among models of one, FP16 storage by
directions and by arcs, all splits of order 2 and none, rows gathered, staged, alone in
a block and too long for one, arcs of one and two tiles, and orders that end at
different levels."""
import numpy as np
import pytest

import parity
import precomputed_atmospheric_scattering_amd as atmo
from precomputed_atmospheric_scattering_amd import configs

pytestmark = pytest.mark.gpu

NAMES = ("transmittance", "scattering", "single_mie_scattering", "irradiance")


def config(tw, r, mu, mu_s, nu, wavelengths=3, half=False):
    z = dict(transmittance_width=tw, transmittance_height=16, scattering_r=r, scattering_mu=mu,
             scattering_mu_s=mu_s, scattering_nu=nu, irradiance_width=16, irradiance_height=4)
    if wavelengths == 3:
        return configs.earth(lut_sizes=z, half_precision=half)
    return configs.spectral(lut_sizes=z, half_precision=half,
                            num_precomputed_wavelengths=wavelengths)


# The models of a batch, each with its orders.
BATCHES = {
    "iterations": [(config(64, 8, 32, 8, 4, 15), 4), (config(64, 8, 32, 8, 4), 2),
                   (config(64, 16, 64, 13, 5, 18), 3), (config(300, 16, 34, 48, 4, 9), 5),
                   (config(4096, 4, 16, 13, 5, 6), 1), (config(64, 3, 22, 9, 16, 6), 4)],
    "storage": [(config(64, 8, 64, 16, 4, 3, True), 4), (config(64, 8, 64, 16, 4, 3), 4),
                (config(64, 5, 46, 9, 7, 15, True), 3), (config(64, 64, 128, 64, 9, 3, True), 3),
                (config(64, 32, 128, 24, 20), 3), (config(64, 2, 4, 2, 2, 3, True), 5)],
    "rows": [(config(256, 16, 50, 32, 8), 3), (config(64, 4, 10, 73, 7, 3, True), 3),
             (config(64, 4, 10, 64, 17, 6), 3), (config(64, 32, 64, 64, 10), 2),
             (config(64, 8, 34, 4, 2, 15, True), 4), (config(64, 41, 70, 9, 3, 15, True), 2)],
}


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("name", sorted(BATCHES))
def test_equals_each_alone(name, use_graph):
    members = BATCHES[name]
    models = [parity.gpu_model(c) for c, _ in members]
    want = []
    for m, (_, orders) in zip(models, members):
        m.init(orders)
        want.append([np.array(m.lut(n)) for n in NAMES])
    b = atmo.Batch(models, [o for _, o in members], use_graph=use_graph)
    for _ in range(2):
        b.launch()
        atmo.synchronize()
        for i, m in enumerate(models):
            for n, w in zip(NAMES, want[i]):
                assert np.array_equal(m.lut(n), w), (i, n)
    b.close()
    for m in models:
        m.close()
