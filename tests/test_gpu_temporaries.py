"""The block of Init temporaries kept between calls of Init: models of different
sizes that take it in turn, from one thread and from several with streams of
their own, have the LUTs of a first Init, bit for bit, and the last model's end
frees it."""
import os
import subprocess
import sys
import threading

import numpy as np
import pytest
import torch

import parity
from precomputed_atmospheric_scattering_amd import configs

pytestmark = pytest.mark.gpu

SIZES = [parity.SMALL_SIZES, parity.MID_SIZES]


def luts(m):
    return [np.array(m.lut(n)) for n in ("transmittance", "scattering", "irradiance")]


def models():
    cfgs = [configs.earth(lut_sizes=SIZES[0]), configs.spectral(lut_sizes=SIZES[0]),
            configs.earth(lut_sizes=SIZES[1], half_precision=True)]
    return [parity.gpu_model(c) for c in cfgs]


def test_blocks_in_turn_and_from_threads():
    ms = models()
    want = []
    for m in ms:
        m.init(3)
        want.append(luts(m))
    for i in (1, 0, 2, 0, 1):  # a smaller model after a larger one
        ms[i].init(3)
        assert all(np.array_equal(a, b) for a, b in zip(luts(ms[i]), want[i]))

    done = []

    def work(i):
        s = torch.cuda.Stream()
        for _ in range(5):
            ms[i].init(3, stream=s.cuda_stream)
        done.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(ms))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert sorted(done) == [0, 1, 2]
    for m, w in zip(ms, want):
        assert all(np.array_equal(a, b) for a, b in zip(luts(m), w))


CHILD = """
import torch
import precomputed_atmospheric_scattering_amd as atmo
from precomputed_atmospheric_scattering_amd import configs
kw, _ = configs.model_kwargs(configs.spectral())
m = atmo.Model(**kw)  # 568 MB of temporaries
m.init(2)
torch.cuda.synchronize()
held = torch.cuda.mem_get_info()[0]
m.close()
print("freed", torch.cuda.mem_get_info()[0] - held)
"""


def test_last_model_frees_it():
    # In a process with no other model. The LUTs are 75 MB.
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, PYTHONPATH=root)
    out = subprocess.run([sys.executable, "-c", CHILD], env=env, capture_output=True,
                         text=True, timeout=100)
    assert out.returncode == 0, out.stderr
    assert int(out.stdout.split()[-1]) > 500e6
