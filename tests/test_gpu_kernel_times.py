"""mpm_kernel_times holds the main kernel of each phase alone."""
import numpy as np
import pytest

from mpm_cuda_amd import capi
from tests.scenes import MAT_PARAMS

pytestmark = pytest.mark.gpu


def _beside(form):
    """Microseconds a step of the grid phase beside its main kernel."""
    h, E_nu_rho = 1.0 / 64, MAT_PARAMS[capi.JELLO]
    s = capi.Sim(capi.default_config(h=h, nx=64, ny=64, nz=64, dt=1e-5, bc_pad=3, form=form, sort_every=1000))
    try:
        x = 0.3 + 0.2 * np.random.default_rng(1).random((20_000, 3))
        s.add_particles(capi.material(*E_nu_rho, capi.JELLO), x.astype(np.float32), volume=h ** 3 / 8)
        s.run(5)
        s.sync()
        s.set_timing(True)
        out = []
        for _ in range(7):
            s.phase_times(), s.kernel_times()
            s.run(20)
            s.sync()
            (phase, n), (kernel, m) = s.phase_times()["grid"], s.kernel_times()["grid"]
            assert n == m == 20
            out.append((phase - kernel) / n * 1e3)
        return float(np.median(out))
    finally:
        s.close()


def test_grid_kernel_alone(gpu):
    """The PLAIN form's grid phase lists the marked blocks first, two launches
    that the FAST form's phase does not have: they are the phase's, not the
    kernel's.  A launch takes at least one microsecond."""
    plain, fast = _beside(capi.FORM_PLAIN), _beside(capi.FORM_FAST)
    print("beside the kernel: plain", plain, "fast", fast)
    assert plain > fast + 2.0
