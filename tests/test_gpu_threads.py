"""Every accepted workgroup size of the particle kernels gives the default's
particles: one group and several, both forms that take it."""
import numpy as np
import pytest

from mpm_cuda_amd import capi
from tests.scenes import MAT_PARAMS, rel

pytestmark = pytest.mark.gpu

N_GRID, STEPS = 32, 6


def _run(form, groups, threads):
    h = 1.0 / N_GRID
    s = capi.Sim(capi.default_config(h=h, nx=N_GRID, ny=N_GRID, nz=N_GRID, dt=1e-4, bc_pad=3, form=form, sort_every=3,
                                     threads=threads))
    try:
        for k in range(groups):
            E, nu, rho = MAT_PARAMS[(capi.JELLO, capi.WATER, capi.SNOW)[k]]
            n = (513, 257, 64)[k]       # not whole workgroups of any size
            x = (np.array([8 + 6 * k, 10, 12]) + 4 * np.random.default_rng(k).random((n, 3))) * h
            s.add_particles(capi.material(E, nu, rho, (capi.JELLO, capi.WATER, capi.SNOW)[k]), x.astype(np.float32),
                            v0=(1.0, -2.0, 0.5), volume=h ** 3 / 8)
        s.run(STEPS)
        return [s.read(k, f) for k in range(groups) for f in (capi.P_POS, capi.P_VEL)]
    finally:
        s.close()


# The parity tests' one-step bounds against 64 bits, once per side and step.
@pytest.mark.parametrize("threads", [64, 128, 256, 512])
@pytest.mark.parametrize("groups", [1, 3])
@pytest.mark.parametrize("form", [capi.FORM_PLAIN, capi.FORM_FAST])
def test_workgroup_sizes(gpu, form, groups, threads):
    for k, (a, b) in enumerate(zip(_run(form, groups, threads), _run(form, groups, 0))):
        assert rel(a, b) < (2e-5 if k % 2 else 2e-6) * STEPS
