"""The launch rules of csrc/kernels.h (which kernel a job takes), compiled for
the host: no GPU needed."""
import itertools
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    """f(jobs) -> per job (block, staged, nit, fixed, lds, fixed_sums, sd_split,
    ms_pairs, ms_spread, arc_sums)."""
    exe = str(tmp_path_factory.mktemp("rules") / "host_rules")
    cxx = shutil.which("amdclang++") or "/opt/rocm/bin/amdclang++"
    r = subprocess.run([cxx, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        os.path.join(HERE, "cpp", "host_rules.cc"), "-o", exe],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr

    def f(jobs):
        text = "\n".join(" ".join(str(int(v)) for v in j) for j in jobs)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, timeout=60)
        rows = [tuple(map(int, l.split())) for l in out.stdout.splitlines()]
        assert out.returncode == 0 and len(rows) == len(jobs)
        return rows
    return f


def job(tw=256, nr=32, nmu=128, nmus=32, nnu=8, niter=1, it=0, half=0, acc64=None):
    return (tw, 64, nr, nmu, nmus, nnu, 64, niter, it, half,
            niter > 1 if acc64 is None else acc64)


ROWS = [(2, 2), (8, 4), (13, 5), (16, 4), (16, 6), (32, 4), (32, 6), (32, 8), (27, 11), (64, 8),
        (64, 16), (512, 32), (4096, 32)]
JOBS = [job(tw, nr, nmu, nmus, nnu, niter)
        for tw, (nr, nmu), (nmus, nnu), niter in itertools.product(
            (2, 64, 256, 512, 1024, 2048, 4096), ((2, 4), (8, 32), (32, 128), (64, 256)), ROWS,
            (1, 2, 5, 7))]


def test_staged_blocks_blend_no_more_than_they_save(rules):
    # A staged block blends TW columns per sample and iteration for its texels; up to
    # 768 blocks of one or two iterations that gather are one round of three per CU.
    staged = 0
    for (tw, _, nr, nmu, nmus, nnu, _, niter, _, _, _), r in zip(JOBS, rules(JOBS)):
        block, stage, nit, _, lds = r[:5]
        w = nmus * nnu
        if stage:
            staged += 1
            assert tw <= (4 if niter > 1 and block > 256 else 2) * block
            assert w >= 160 and lds <= 64 << 10
            gathering = nr * nmu * -(-w // 256)
            assert gathering >= 512 and (niter > 2 or gathering > 768)
        else:
            assert lds == 0 and block <= 256
        assert block >= 64 and nit in (1, niter if niter < 5 else 5)
    assert 0 < staged < len(JOBS)


def test_staged_blocks_fit_their_rows(rules):
    # Rows of 513..768 texels take 256-thread blocks; 2 columns a thread, or 4 in
    # blocks of 512 that serve several iterations.
    jobs = [job(nmus=w // 4, nnu=4, tw=tw, niter=n) for w, tw, n in (
        (156, 256, 1), (160, 256, 1), (192, 512, 1), (256, 512, 1), (256, 513, 5), (260, 1024, 1),
        (260, 1025, 1), (260, 2048, 2), (512, 512, 1), (516, 512, 1), (768, 512, 5),
        (768, 513, 5), (772, 512, 1))]
    assert [r[:2] for r in rules(jobs)] == [
        (256, 0), (256, 1), (256, 0), (256, 1), (256, 0), (512, 1), (256, 0), (512, 1), (512, 1),
        (256, 1), (256, 1), (512, 1), (512, 1)]
    # 768 and 780 blocks of 256; 510 and 512.
    jobs = [job(nr=16, nmu=48), job(nr=15, nmu=52), job(nr=15, nmu=34, niter=5),
            job(nr=16, nmu=32, niter=5), job(nr=16, nmu=32, niter=2)]
    assert [r[1] for r in rules(jobs)] == [0, 1, 0, 1, 0]


def test_iterations_are_served_once(rules):
    # The blocks of an iteration serve the nit - 1 that follow it.
    for tw, nmus in itertools.product((64, 1024, 4096), (4, 32)):
        for niter in range(1, 12):
            rs = rules([job(tw, nmus=nmus, niter=niter, it=i) for i in range(niter)])
            i = 0
            while i < niter:
                nit = rs[i][2]
                assert 1 <= nit <= 5 and i + nit <= niter
                assert all(rs[k][2] == 0 for k in range(i + 1, i + nit))
                assert all(rs[k][:2] == rs[i][:2] for k in range(i, i + nit))
                i += nit


def test_few_blocks_load_texel_by_texel(rules):
    # Rows of 256 texels, one per block of one-texel threads; rows of 96 at any size.
    assert [r[7] for r in rules([job(nr=8, nmu=32, half=1), job(nr=32, nmu=64, half=1),
                                 job(nr=31, nmu=66, half=1), job(nr=16, nmu=26, niter=5, half=1),
                                 job(nr=32, nmu=128), job(nr=2, nmu=4, nmus=64, half=1),
                                 job(nr=64, nmu=256, nmus=16, nnu=6, niter=5, half=1)])] == [
        0, 1, 0, 1, 0, 1, 0]
    # FP32 rows of 640 alone in a block.
    assert [r[8] for r in rules([job(nr=8, nmu=32, nmus=64, nnu=10),
                                 job(nr=8, nmu=34, nmus=64, nnu=10),
                                 job(nr=2, nmu=24, nmus=64, nnu=10, niter=5),
                                 job(nr=2, nmu=26, nmus=64, nnu=10, niter=5),
                                 job(nr=8, nmu=32, nmus=64, nnu=10, half=1), job(nr=2, nmu=4)])
            ] == [1, 0, 1, 0, 0, 0]


def test_arc_sums(rules):
    # 3 wavelengths: NU 20 and more from 1.9M texels on take the directions; so do
    # FP16-storage models of up to 2^22 texels.
    jobs = [job(nr=64, nmu=256, nmus=64, nnu=16), job(nr=32, nmu=128, nmus=32, nnu=19),
            job(nr=32, nmu=128, nmus=32, nnu=20), job(nr=32, nmu=128, nmus=20, nnu=23),
            job(nr=32, nmu=128, nmus=20, nnu=24), job(nr=32, nmu=128, nmus=20, nnu=32, niter=2),
            job(nr=32, nmu=128, half=1), job(nr=64, nmu=128, nmus=64, nnu=8, half=1),
            job(nr=64, nmu=128, nmus=64, nnu=9, half=1), job(nr=64, nmu=128, nmus=64, half=1,
                                                             nnu=20)]
    got = rules(jobs)
    assert [r[9] for r in got] == [1, 1, 0, 1, 0, 1, 0, 0, 1, 0]
    # What is summed by directions at the orders >= 3 has a thread per output.
    assert all(r[6] == 3 for r in got if not r[9])
