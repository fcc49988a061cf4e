"""Several particle groups in one launch, and the list of grid blocks kept
between sorts: the FAST form against the PLAIN one (a launch per group, the
marked blocks listed at every step) on the same state."""
import numpy as np
import pytest

from mpm_cuda_amd import capi
from tests.scenes import MAT_PARAMS, rel

pytestmark = pytest.mark.gpu

N_GRID, DT, STEPS = 64, 1e-4, 12
SIZES = [300, 1, 64, 257, 63, 500, 129, 65, 255, 400]
TYPES = [capi.JELLO, capi.WATER, capi.SNOW]


def _sim(form, sizes, same, cells_per_step, **cfg):
    h = 1.0 / N_GRID
    sim = capi.Sim(capi.default_config(h=h, nx=N_GRID, ny=N_GRID, nz=N_GRID, dt=DT, bc_pad=3, form=form,
                                       sort_every=50, **cfg))
    rng = np.random.default_rng(len(sizes))
    for k, n in enumerate(sizes):
        type_ = TYPES[0 if same else k % 3]
        E, nu, rho = MAT_PARAMS[type_]
        side = max(1.0, (n / 4.0) ** (1 / 3))
        x = (np.array([14 + 9 * (k % 4), 16 + 9 * (k // 4), 30 + k % 3]) + side * rng.random((n, 3))) * h
        way = np.array([[1, -1, 1], [-1, 1, 0.5], [0.3, 1, -1]][k % 3])
        sim.add_particles(capi.material(E, nu, rho, type_), x.astype(np.float32),
                          v0=tuple(cells_per_step * way * h / DT), volume=h ** 3 / 4)
    return sim


# Bounds: the parity tests' one-step bounds against 64 bits (x 1e-6, the
# rest 1e-5), once per form and step.
@pytest.mark.parametrize("ngroups,same", [(1, True), (2, False), (8, True), (9, False), (10, True)])
@pytest.mark.parametrize("cells_per_step", [0.0, 0.15], ids=["rest", "fast"])
@pytest.mark.parametrize("cfl", [False, True], ids=["fixed", "cfl"])
def test_groups_and_block_list(gpu, ngroups, same, cells_per_step, cfl):
    extra = dict(dt_mode=capi.DT_CFL, cfl=0.5) if cfl else {}
    fast = _sim(capi.FORM_FAST, SIZES[:ngroups], same, cells_per_step, **extra)
    plain = _sim(capi.FORM_PLAIN, SIZES[:ngroups], same, cells_per_step, **extra)
    try:
        spilled = 0
        for k in range(STEPS):
            fast.step()
            plain.step()
            a, b = fast.stats(), plain.stats()
            spilled = max(spilled, a["spilled"])
            tol = 2e-5 * (k + 1)
            assert a["active_blocks"] == b["active_blocks"], k
            assert rel(fast.grid(capi.G_MASS), plain.grid(capi.G_MASS)) < tol
            assert rel(fast.grid(capi.G_VELOCITY) * fast.grid(capi.G_MASS)[..., None],
                       plain.grid(capi.G_VELOCITY) * plain.grid(capi.G_MASS)[..., None]) < tol
        for g in range(ngroups):
            assert rel(fast.read(g, capi.P_POS), plain.read(g, capi.P_POS)) < 2e-6 * STEPS
            assert rel(fast.read(g, capi.P_VEL), plain.read(g, capi.P_VEL)) < 2e-5 * STEPS
        assert (spilled > 0) == (cells_per_step > 0)    # drifted out of the blocks of the only sort so far
        assert abs(fast.current_time - plain.current_time) <= 1e-6 * plain.current_time
    finally:
        fast.close()
        plain.close()


@pytest.mark.parametrize("type_", TYPES)
def test_batch_of_one_material(gpu, type_):
    """Scenes of a single material advanced as a batch and one by one."""
    sims, alone = [], []
    E, nu, rho = MAT_PARAMS[type_]
    for out in (sims, alone):
        for k, n in enumerate((257, 1)):
            s = capi.Sim(capi.default_config(h=1.0 / N_GRID, nx=N_GRID, ny=N_GRID, nz=N_GRID, dt=DT, bc_pad=3,
                                             form=capi.FORM_FAST))
            x = 0.4 + 0.08 * np.random.default_rng(k).random((n, 3))
            s.add_particles(capi.material(E, nu, rho, type_), x.astype(np.float32), v0=(1.0, -2.0, 0.5),
                            volume=0.25 / N_GRID ** 3)
            out.append(s)
    batch = capi.Batch(sims, capi.batch_shape(sort_every=3))
    try:
        batch.run(7)
        batch.sync()
        for s, a in zip(sims, alone):
            a.run(7)
            assert s.stats()["active_blocks"] == a.stats()["active_blocks"]
            assert rel(s.read(0, capi.P_POS), a.read(0, capi.P_POS)) < 2e-6 * 7
            assert rel(s.read(0, capi.P_VEL), a.read(0, capi.P_VEL)) < 2e-5 * 7
    finally:
        batch.close()
        for s in sims + alone:
            s.close()
