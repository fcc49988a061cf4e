"""Batches that step as two chains of launches side by side: the same particles
as scenes stepped alone, and a step shorter than the sum of its stages."""
import numpy as np
import pytest

from mpm_cuda_amd import capi, warm_start, workloads
from tests.scenes import rel

pytestmark = pytest.mark.gpu


def _scenes(sizes, **cfg):
    mats = (capi.JELLO, capi.SNOW, capi.WATER)
    return [workloads.batch_scene(mats[k % 3], 96, n, 50 + k, **cfg)[0] for k, n in enumerate(sizes)]


def _same(sims, alone, steps):
    """The parity tests' bounds against 64 bits, once per side and step."""
    for s, a in zip(sims, alone):
        assert s.current_frame == a.current_frame
        assert rel(s.read(0, capi.P_POS), a.read(0, capi.P_POS)) < 2e-6 * steps
        assert rel(s.read(0, capi.P_VEL), a.read(0, capi.P_VEL)) < 2e-5 * steps


# 200,000 particles are the least that take chains; a scene that is more than
# half of them, two scenes, and runs below and from the least number of steps
@pytest.mark.parametrize("sizes", [(100_000, 100_001), (20_000, 150_000, 31_000, 1_000), (40_000,) * 6],
                         ids=["two", "uneven", "six"])
@pytest.mark.parametrize("timed", [False, True])
def test_chains_match_single_scenes(gpu, sizes, timed):
    sims, alone = _scenes(sizes), _scenes(sizes)
    batch = capi.Batch(sims, capi.batch_shape(sort_every=5))
    try:
        assert batch.particles >= 200_000
        for n in (12, 1, 11, 13):
            ms = batch.run(n, timed=timed)
            assert not timed or (ms.shape == (n,) and np.all(ms > 0))
        sims[1].run(2)                  # on its own stream, after the chains
        batch.run(12)
        batch.sync()
        for k, a in enumerate(alone):
            a.run(51 if k == 1 else 49)
        _same(sims, alone, 51)
    finally:
        batch.close()
        for s in sims + alone:
            s.close()


def test_chains_with_warm_start(gpu):
    """Two weight sets, so that a chain may hold either or both."""
    w = warm_start.load_weights()
    w2 = (w + 0.01 * np.random.default_rng(40).normal(size=w.size)).astype(np.float32)
    kw = dict(warm_start=capi.WARM_MLP, warm_sweeps=2)
    sims, alone = _scenes((60_000,) * 5, **kw), _scenes((60_000,) * 5, **kw)
    for k, s in enumerate(sims + alone):
        s.set_warm_start_weights(w2 if k % 5 in (1, 3) else w)
        F = np.tile(np.eye(3, dtype=np.float32).reshape(9), (s.total, 1))
        F[::3, 0] = 0.95 if k % 5 % 3 == 1 else 2.2     # outside the cheap path's band
        s.write(0, capi.P_F, F)
    batch = capi.Batch(sims, capi.batch_shape(sort_every=50))
    try:
        batch.run(12)
        batch.sync()
        for a in alone:
            a.run(12)
        _same(sims, alone, 12)
        for k, (s, a) in enumerate(zip(sims, alone)):
            if k % 3 != 2:
                sa, sb = s.svd_stats(), a.svd_stats()
                assert sa["svd"] > 0 and sa["warm"] > 0.5 * sa["svd"] and sb["warm"] > 0.5 * sb["svd"]
    finally:
        batch.close()
        for s in sims + alone:
            s.close()


def test_stages_of_two_halves_overlap(gpu):
    """24 scenes, 1.7M particles: a step's median is below 0.94 of the sum of
    the stages' (0.88 with two chains, 0.97 with one).  The best of five runs,
    since the clock is shared with whatever else the machine does."""
    sims = _scenes((70_000,) * 24)
    batch = capi.Batch(sims)
    try:
        best = []
        for _ in range(5):
            tune = batch.autotune(reps=2)
            stages = sum(min(tune[k].values()) for k in ("p2g", "grid", "g2p"))
            best.append(float(np.median(batch.run(48, timed=True))) / stages)
        print("step over stages", best)
        assert min(best) < 0.94
    finally:
        batch.close()
        for s in sims:
            s.close()
