"""Particle reads: every field comes back in particle-id order, bit for bit,
at the sizes where the transfer takes another form."""
import threading

import numpy as np
import pytest

from mpm_cuda_amd import capi

pytestmark = pytest.mark.gpu

# 1 MiB of positions is 87381.3 rows, of F 29127.1; 4 MiB of positions 349525.3
SIZES = [1, 255, 257, 29127, 29128, 87381, 87382, 349526, 700001]


def _sim(n, seed=0):
    rng = np.random.default_rng(seed)
    sim = capi.Sim(capi.default_config(nx=96, ny=96, nz=96, h=1 / 96, dt=1e-5))
    x = (0.2 + 0.6 * rng.random((n, 3))).astype(np.float32)
    sim.add_particles(capi.material(5e4, 0.3, 1e3, capi.JELLO), x, volume=1e-6)
    return sim, rng


@pytest.mark.parametrize("n", SIZES)
def test_read_returns_what_was_written(gpu, n):
    sim, rng = _sim(n)
    try:
        sim.run(3)          # sorted: stored in another order than the ids'
        for field, w in ((capi.P_POS, 3), (capi.P_VEL, 3), (capi.P_C, 9), (capi.P_F, 9), (capi.P_JP, 1)):
            a = (0.2 + 0.6 * rng.random((n, w))).astype(np.float32)
            sim.write(0, field, a)
            for _ in range(2):
                assert np.array_equal(sim.read(0, field), a)
        assert np.array_equal(sim.positions(), sim.read(0, capi.P_POS))
    finally:
        sim.close()


@pytest.mark.parametrize("n", [1000, 200_003, 600_000])
def test_2d_read_returns_what_was_added(gpu, n):
    rng = np.random.default_rng(1)
    sim = capi.Sim2D(n_grid=128)
    x, v = (0.2 + 0.6 * rng.random((n, 2))).astype(np.float32), rng.normal(size=(n, 2)).astype(np.float32)
    sim.add_particles(x, v)
    assert np.array_equal(sim.read(capi.P2_POS), x) and np.array_equal(sim.read(capi.P2_VEL), v)
    assert np.array_equal(sim.read(capi.P2_F), np.tile(np.float32([1, 0, 0, 1]), (n, 1)))


def test_reads_from_two_threads(gpu):
    sim, _ = _sim(120_000)
    try:
        sim.run(2)
        want = {f: sim.read(0, f) for f in (capi.P_POS, capi.P_VEL)}
        bad = []

        def work(field):
            for _ in range(20):
                if not np.array_equal(sim.read(0, field), want[field]):
                    bad.append(field)

        threads = [threading.Thread(target=work, args=(f,)) for f in want]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not bad
    finally:
        sim.close()
