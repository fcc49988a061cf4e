"""FAST-form P2G over tiles of every awkward size against the FP64 oracle."""
import numpy as np
import pytest

from mpm_cuda_amd import capi
from tests import scenes
from tests.scenes import Pair, rel

pytestmark = pytest.mark.gpu

# particles of the tiles: around one, two and four waves and the passes of
# each; on average above and below the count that chooses the wide workgroup
DENSE = [1, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 513, 769]
SPARSE = [1, 2, 31, 63, 64, 65, 100, 127, 128, 129, 1, 193, 257]
N_GRID, BLK = 64, 4


def _tiles(counts, one_cell, seed):
    """counts[k] particles in the k-th of a row of separate node blocks, over
    the block's cells or all in its last one."""
    rng = np.random.default_rng(seed)
    out = []
    for k, c in enumerate(counts):
        origin = np.array([2 + 2 * (k % 6), 4 + 3 * (k // 6), 5 + k % 3]) * BLK
        rel_pos = BLK - 1 + rng.random((c, 3)) if one_cell else BLK * rng.random((c, 3))
        out.append(origin + 0.5 + np.minimum(rel_pos, BLK - 1e-4))
    return (np.concatenate(out) / N_GRID).astype(np.float32)


# Grid spacing a power of two: positions relative to the base node are exact,
# so a mass carries the roundings of three weights and two products (about ten
# of 2^-24); the momentum bar is the parity tests' (FP32 stress included).
@pytest.mark.parametrize("type_", [capi.JELLO, capi.SNOW, capi.WATER])
@pytest.mark.parametrize("counts,one_cell,fast", [(DENSE, False, 1.0), (SPARSE, False, 1.0), (SPARSE, True, 1.0),
                                                  (DENSE, False, 300.0)],
                         ids=["dense", "sparse", "one-cell", "one-fast"])
def test_p2g_tile_sizes(gpu, monkeypatch, type_, counts, one_cell, fast):
    x = _tiles(counts, one_cell, 5)
    monkeypatch.setattr(scenes, "jittered_box", lambda *a: x)
    p = Pair(type_=type_, form=capi.FORM_FAST, n_grid=N_GRID, seed=3)
    try:
        v = p.gpu.read(0, capi.P_VEL)
        v[::97] *= fast                 # the tile's scale is that of its fastest particle
        p.gpu.write(0, capi.P_VEL, v)
        p.orc.groups[0].v[:] = v
        p.orc.clear_grid()
        assert p.orc.p2g(p.dt) == 0
        first = None
        for _ in range(3):              # the first before the width is known, the same sums after
            p.gpu.phase(capi.PHASE_P2G, p.dt)
            m, mom = p.gpu.grid(capi.G_MASS), p.gpu.grid(capi.G_MOMENTUM)
            assert rel(m, p.orc.grid_mass()) < 1e-6
            assert rel(mom, p.orc.grid_vec()) < 1e-5
            if first is None:
                first = m, mom
            assert np.array_equal(first[0], m) and np.array_equal(first[1], mom)
        assert p.gpu.stats()["tiles"] == len(counts)
    finally:
        p.close()


@pytest.mark.parametrize("gamma", [1.0, 2.0, 7.0, 32.0, 33.0, 2.5, 0.5])
@pytest.mark.parametrize("form", [capi.FORM_PLAIN, capi.FORM_FAST])
def test_water_pressure_exponents(gpu, form, gamma):
    """Whole exponents (products) and others (powf); the parity tests' bar."""
    p = Pair(type_=capi.WATER, form=form, seed=4, eos_gamma=gamma)
    try:
        p.gpu.phase(capi.PHASE_P2G, p.dt)
        p.orc.clear_grid()
        assert p.orc.p2g(p.dt) == 0
        assert rel(p.gpu.grid(capi.G_MOMENTUM), p.orc.grid_vec()) < 1e-5
    finally:
        p.close()
