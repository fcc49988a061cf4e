"""FAST-form P2G where the particles of one tile, or the components of their
velocities, differ by many orders of magnitude in speed or pressure: every
node keeps the accuracy of FP32 sums of its own contributions, whatever else
the tile holds."""
import numpy as np
import pytest

from mpm_cuda_amd import capi
from tests.scenes import MAT_PARAMS

pytestmark = pytest.mark.gpu

N_GRID, BLK, DT, COUNT = 64, 4, 1e-4, 500
H = 1.0 / N_GRID
EOS_K = 1e4
ORIGIN = np.array([5, 6, 7]) * BLK

# Bars at every node.  The grid spacing is a power of two and positions are
# multiples of 2^-10 cells, so offsets from nodes are exact; a contribution
# carries about 20 roundings of 2^-24 (three weights and their products, the
# affine and the force term, the pressure) and a sum up to four more.  Adding a
# contribution to a tile's sums may cost 2^-26 of the bound on that particle's
# contributions (where all of a tile's particles are alike in a component, of
# that component's bound); a mass 2^-41 of the particle's (COUNT is below 2^9).
TOL, TOL_ADD = 24 * 2.0 ** -24, 2.0 ** -26
TOL_MASS, TOL_MASS_ADD = 12 * 2.0 ** -24, 2.0 ** -41


def _positions(rng):
    """COUNT particles with their base nodes in the block at ORIGIN."""
    cells = rng.integers(0, BLK, (COUNT, 3)) + rng.integers(0, 1024, (COUNT, 3)) / 1024.0
    return ORIGIN + 0.5 + cells


def _state(type_, kind, ratio, seed):
    """(x in cells, v, C, J): ordinary particles, and those that `kind` makes
    large: the last one, by its speed or its J, half of them, or a layer of
    cells in x each `ratio` times as fast as the one before; or all of them
    `ratio` times slower along x ("flat")."""
    rng = np.random.default_rng(seed)
    x = _positions(rng)
    v = rng.uniform(0.5, 1.0, (COUNT, 3)) * rng.choice([-1.0, 1.0], (COUNT, 3))
    C = rng.uniform(-20.0, 20.0, (COUNT, 9))
    J = np.ones(COUNT)
    v[::50] = 0.0                        # and some that carry mass only
    C[::50] = 0.0
    if kind == "layers":
        x[:, 0] = ORIGIN[0] + 0.5 + np.arange(COUNT) % 4 + rng.integers(0, 1024, COUNT) / 1024.0
        s = ratio ** np.floor(x[:, 0] - ORIGIN[0] - 0.5)
        v *= s[:, None]
        C *= s[:, None]
    elif kind == "flat":
        v[:, 0] /= ratio
        C[:, :3] /= ratio
    elif kind == "half":
        v[COUNT // 2:] *= ratio
        C[COUNT // 2:] *= ratio
    else:
        x[-1] = ORIGIN + 3.5 + 0.25      # in the block's last cell
        if kind == "J":
            J[-1] = ratio
        else:
            v[-1] = ratio * np.array([0.7, -0.5, 0.6])
    f = np.float32
    return x, v.astype(f), C.astype(f), J.astype(f)


def _reference(sim, type_, x, v, C, J):
    """64-bit nodes of the tile: mass, momentum, sum of the contributions'
    magnitudes, and of the particles that reach the node the sum of the bounds
    on their contributions and their mass."""
    rho = MAT_PARAMS[type_][2]
    vol = float(np.float32(H ** 3 / 8))
    m = float(np.float32(rho * H ** 3 / 8))
    dt = float(np.float32(DT))
    v, C, J = v.astype(np.float64), C.reshape(-1, 3, 3).astype(np.float64), J.astype(np.float64)
    if type_ == capi.WATER:
        G = (dt * vol * EOS_K * (J ** -7 - 1) * J)[:, None, None] * np.eye(3)
    else:
        xx, yy, zz, xy, xz, yz = sim.read(0, capi.P_TAU).astype(np.float64).T
        G = -dt * vol * np.stack([xx, xy, xz, xy, yy, yz, xz, yz, zz], -1).reshape(-1, 3, 3)
    base = np.floor(x - 0.5).astype(int)
    fx = x - base
    N = np.stack([0.5 * (1.5 - fx) ** 2, 0.75 - (fx - 1) ** 2, 0.5 * (fx - 0.5) ** 2], 1)     # [p][o][axis]
    D = np.stack([fx - 1.5, -2 * (fx - 1), fx - 0.5], 1) / H
    bound = (np.abs(v) * m + 3.5 * H * m * np.abs(C).sum(2) + np.abs(G).sum(2) / H)
    out = np.zeros((5, N_GRID, N_GRID, N_GRID, 3))
    mass, mom, mag, bnd, reach = out
    for o in np.ndindex(3, 3, 3):
        w = N[:, o[0], 0] * N[:, o[1], 1] * N[:, o[2], 2]
        gw = np.stack([D[:, o[0], 0] * N[:, o[1], 1] * N[:, o[2], 2], N[:, o[0], 0] * D[:, o[1], 1] * N[:, o[2], 2],
                       N[:, o[0], 0] * N[:, o[1], 1] * D[:, o[2], 2]], 1)
        d = (np.array(o) - fx) * H
        affine = np.einsum("pck,pk->pc", C, d)
        force = np.einsum("pck,pk->pc", G, gw)
        at = tuple((base + o)[:, k] for k in (2, 1, 0))
        np.add.at(mass, at, (w * m)[:, None])
        np.add.at(mom, at, (w * m)[:, None] * (v + affine) + force)
        np.add.at(mag, at, (w * m)[:, None] * (np.abs(v) + np.einsum("pck,pk->pc", np.abs(C), np.abs(d))) +
                  np.einsum("pck,pk->pc", np.abs(G), np.abs(gw)))
        np.add.at(bnd, at, bound)
        np.add.at(reach, at, m)
    return mass[..., 0], mom, mag, bnd, reach[..., 0]


def _sim(type_, x, v, C, J):
    E, nu, rho = MAT_PARAMS[type_]
    s = capi.Sim(capi.default_config(h=H, nx=N_GRID, ny=N_GRID, nz=N_GRID, dt=DT, bc_pad=3, form=capi.FORM_FAST))
    s.add_particles(capi.material(E, nu, rho, type_, eos_k=EOS_K, eos_gamma=7.0), (x * H).astype(np.float32),
                    volume=H ** 3 / 8)
    s.write(0, capi.P_VEL, v)
    s.write(0, capi.P_C, C)
    if type_ == capi.WATER:
        s.write(0, capi.P_JP, J[:, None])
    return s


def _bar(kind, mag, bnd):
    """What a momentum may be off by, per component: of all components'
    magnitudes and bounds, or ("flat") of its own."""
    if kind != "flat":
        mag, bnd = mag.sum(-1, keepdims=True), bnd.sum(-1, keepdims=True)
    return TOL * mag + TOL_ADD * bnd


CASES = [("flat", 2.0 ** 30), ("v", 2.0 ** 10), ("v", 2.0 ** 20), ("v", 2.0 ** 30), ("half", 2.0 ** 20), ("layers", 2.0 ** 16),
         ("J", 0.5), ("J", 0.1), ("J", 0.02)]


@pytest.mark.parametrize("type_,kind,ratio", [(t, k, r) for t in (capi.JELLO, capi.SNOW, capi.WATER) for k, r in CASES
                                              if k != "J" or t == capi.WATER])
def test_tile_of_a_wide_range(gpu, type_, kind, ratio):
    x, v, C, J = _state(type_, kind, ratio, 3)
    s = _sim(type_, x, v, C, J)
    try:
        mass, mom, mag, bnd, reach = _reference(s, type_, x, v, C, J)
        first = None
        for _ in range(3):
            s.phase(capi.PHASE_P2G, DT)
            gm, gp = s.grid(capi.G_MASS).astype(np.float64), s.grid(capi.G_MOMENTUM).astype(np.float64)
            if first is None:
                first = gm, gp
            assert np.array_equal(first[0], gm) and np.array_equal(first[1], gp)
        over_m = np.abs(gm - mass) - (TOL_MASS * mass + TOL_MASS_ADD * reach)
        over_p = np.abs(gp - mom) - _bar(kind, mag, bnd)
        assert (gm > 0).sum() > 200
        assert over_m.max() <= 0
        worst = np.unravel_index(np.argmax(over_p), over_p.shape)
        assert over_p.max() <= 0, (worst, gp[worst], mom[worst], mag[worst], bnd[worst])
        s.phase(capi.PHASE_GRID, DT)
        assert s.stats()["spilled"] == 0
    finally:
        s.close()


@pytest.mark.parametrize("type_,kind,ratio", [(capi.JELLO, "layers", 2.0 ** 16), (capi.WATER, "J", 0.02)])
def test_batched_tile_of_a_wide_range(gpu, type_, kind, ratio):
    """The batched P2G, from the velocities that the step leaves on the grid
    (a quotient, gravity and their inverses: eight more roundings)."""
    args = _state(type_, kind, ratio, 4)
    s = _sim(type_, *args)
    mass, mom, mag, bnd, _ = _reference(s, type_, *args)
    batch = capi.Batch([s])
    try:
        batch.run(1)
        batch.sync()
        g = DT * np.array([0.0, -9.8, 0.0])
        gp = (s.grid(capi.G_VELOCITY).astype(np.float64) - g * (mass > 0)[..., None]) * mass[..., None]
        over = np.abs(gp - mom) - _bar(kind, mag, bnd) - 8 * 2.0 ** -24 * (mag.sum(-1) + 1e-3 * mass)[..., None]
        sure = mass > 2.0 ** -16 * mass.max()       # where the mass is not itself a few units of its sum
        assert sure.sum() > 200
        assert over[sure].max() <= 0
    finally:
        batch.close()
        s.close()
