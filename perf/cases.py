"""Timing cases of the simulator: what a user's program does with it.

A case is a dict of plain values.  ``listed()`` names the fixed ones,
``draw(rng)`` gives further ones of the same ranges, ``prepare`` builds the
handles a program holds before the call, ``run`` is one pass through the
public entry points (some steps, then the read a program makes of the
result), ``work`` counts what a pass cannot do without, and ``exact`` is the
same pass in 64 bits in plain torch, without this package's code.

Kinds of case:

* ``scene``   -- one simulator in the default (FAST) form: bodies of jello,
  snow or water, or one of each (three particle groups on one grid), `steps`
  time steps and a read: ``positions`` (a rendered or dumped frame), ``viewer``
  (positions and velocities) or ``state`` (every field, a checkpoint).
* ``batch``   -- scenes of several sizes and materials advanced together, the
  positions of each read at the end.
* ``snow2d``  -- the 2D snow simulator, `steps` steps and a read of its state.

Bodies are sampled as the package's own sampler does: whole cells, a fixed
number of jittered samples in each, trimmed to the count asked for.  They
start with a smooth velocity field (drift, spin and long waves drawn from the
seed), so that the affine velocities and the deformation are those of a body
in motion.
"""
import math

import numpy as np
import torch

from mpm_cuda_amd import capi

TYPES = {"jello": capi.JELLO, "snow": capi.SNOW, "water": capi.WATER}
# materials of the package's workloads
PARAMS = {
    "jello": dict(E=5e4, nu=0.3, rho=1e3, extra={}),
    "snow": dict(E=1.4e5, nu=0.2, rho=400.0, extra=dict(theta_c=2.5e-2, theta_s=7.5e-3, xi=10.0)),
    "water": dict(E=1e4, nu=0.2, rho=1e3, extra=dict(eos_k=1e4, eos_gamma=7.0, water_c_mode=capi.WATER_C_GRADV)),
}
STATE = {"jello": ("x", "v", "C", "F"), "snow": ("x", "v", "C", "F", "J"), "water": ("x", "v", "C", "J")}
FIELD = {"x": capi.P_POS, "v": capi.P_VEL, "C": capi.P_C, "F": capi.P_F, "J": capi.P_JP}
FLOATS = {"x": 3, "v": 3, "C": 9, "F": 9, "J": 1}
CFL = 0.5
BATCH_GRIDS = (64, 80, 96, 112, 128, 144, 160)


def listed():
    return [
        # a viewer on a small scene: the reference copies the positions to
        # the host after every step, so one step and its read is a pass
        dict(name="viewer_jello_10k", kind="scene", material="jello", n=10_000, nx=64, ny=64, nz=64, per_cell=8.0,
             dt=1e-4, steps=1, cfl=False, read="viewer"),
        # a small snow scene of the size of the parity tests, its whole state kept
        dict(name="state_snow_16k", kind="scene", material="snow", n=16_000, nx=64, ny=64, nz=64, per_cell=8.0,
             dt=1e-4, steps=10, cfl=False, read="state"),
        # a dam break on a grid whose sides are no multiple of a block
        dict(name="state_water_47k", kind="scene", material="water", n=47_351, nx=81, ny=67, nz=93, per_cell=4.0,
             dt=1e-4, steps=20, cfl=False, read="state"),
        # fast snow under the step-size controller, which it needs
        dict(name="cfl_snow_100k", kind="scene", material="snow", n=100_000, nx=96, ny=96, nz=96, per_cell=8.0,
             dt=1e-4, steps=50, cfl=True, read="positions"),
        # several objects of different materials on one grid, as the
        # reference's scenes have
        dict(name="objects_300k", kind="scene", material="mixed", n=300_000, nx=128, ny=128, nz=128, per_cell=8.0,
             dt=5e-5, steps=50, cfl=False, read="positions"),
        # frames of the three 3D workloads, 100 steps each (the snow at a dt
        # that its hardened state bears)
        dict(name="jello_262k", kind="scene", material="jello", n=262_144, nx=128, ny=128, nz=128, per_cell=8.0,
             dt=1e-4, steps=100, cfl=False, read="positions"),
        dict(name="snow_1m", kind="scene", material="snow", n=1_000_000, nx=192, ny=192, nz=192, per_cell=5.0,
             dt=2.5e-5, steps=100, cfl=False, read="positions"),
        dict(name="water_2m", kind="scene", material="water", n=2_000_000, nx=256, ny=256, nz=256, per_cell=1.2,
             dt=5e-5, steps=100, cfl=False, read="positions"),
        # many scenes at once, for collecting data
        dict(name="batch_16", kind="batch", scenes=16, n_min=10_000, n_max=100_000, steps=48),
        # the reference's 2D snow
        dict(name="snow2d_9k", kind="snow2d", n=9_000, n_grid=128, dt=1e-4, steps=50),
    ]


def draw(rng):
    """One more case: sizes spread over the logarithm of the range, odd ones
    among them, none dearer than the largest listed one."""
    pick = rng.random()
    if pick < 0.12:
        lo = int(10 ** rng.uniform(3.7, 4.5))
        return dict(kind="batch", scenes=rng.randint(2, 20), n_min=lo, n_max=int(lo * rng.uniform(1.5, 8.0)),
                    steps=rng.randint(5, 60))
    if pick < 0.27:
        grid = rng.choice((64, 96, 128, 160, 200, 256))
        n = int(grid * grid * 10 ** rng.uniform(-1.0, 0.4))
        return dict(kind="snow2d", n=max(n, 500), n_grid=grid, dt=1e-4 * min(1.0, 128.0 / grid),
                    steps=rng.randint(1, 120))
    material = rng.choice(("jello", "snow", "water", "mixed", "snow", "jello", "water"))
    n = int(10 ** rng.uniform(3.5, 6.15)) | rng.randint(0, 1)
    per_cell = rng.choice((1.2, 2.0, 4.0) if material == "water" else (4.0, 5.0, 8.0))
    while True:
        need = _extent(material, n, per_cell)
        if max(need) <= 248:
            break
        n //= 2
    nx, ny, nz = (min(256, max(32, m + rng.randint(2, 48))) for m in need)
    read = rng.choice(("positions", "viewer", "state") if n <= 60_000 else ("positions", "viewer"))
    steps = rng.randint(1, 12) if read != "positions" else int(10 ** rng.uniform(0.0, 2.0))
    cfl = material == "snow" and rng.random() < 0.3
    return dict(kind="scene", material=material, n=n, nx=nx, ny=ny, nz=nz, per_cell=per_cell,
                dt=_dt("jello" if cfl else material, max(nx, ny, nz)), steps=steps, cfl=cfl, read=read)


def _dt(material, nodes):
    """A dt that the material bears on a grid of 1 / nodes spacing: compacted
    snow carries waves many times faster than fresh snow."""
    if material in ("snow", "mixed"):
        return min(1e-4, 0.0048 / nodes)
    return 5e-5 if material == "water" and nodes > 96 else 1e-4


# ---------------------------------------------------------------------------
# Bodies.

def _pad(nx, ny, nz):
    return 10 if min(nx, ny, nz) >= 128 else 3


def _shapes(material, n, per_cell):
    """(material, count, ball, sides in cells) of every body, left to right."""
    if material == "mixed":
        third = n // 3
        return (_shapes("jello", third, per_cell) + _shapes("water", third, per_cell) +
                [_ball("snow", n - 2 * third, per_cell)])
    if material == "snow":
        return [_ball("snow", n // 2, per_cell), _ball("snow", n - n // 2, per_cell)]
    cells = n / per_cell
    if material == "jello":
        return [("jello", n, False, (int(math.ceil(cells ** (1 / 3))),) * 3)]
    a = (cells / 0.8) ** (1 / 3)                     # 0.5 : 0.4 : 0.5, the dam break's block
    return [("water", n, False, (int(math.ceil(a)), int(math.ceil(0.8 * a)), int(math.ceil(a))))]


def _ball(material, n, per_cell):
    r = (n / per_cell * 3 / (4 * math.pi)) ** (1 / 3) * 1.02 + 0.3
    return (material, n, True, (int(math.ceil(2 * r)),) * 3)


def _extent(material, n, per_cell):
    """Nodes per axis that hold the bodies between 10-cell walls."""
    s = _shapes(material, n, per_cell)
    return (sum(b[3][0] + 2 for b in s) + 28, max(b[3][1] for b in s) + 28, max(b[3][2] for b in s) + 28)


def _sample(rng, n, per_cell, ball, sides):
    """n points of a body in cells from its corner: ceil(per_cell) jittered
    samples in every cell, trimmed to n."""
    k = max(1, int(math.ceil(per_cell)))
    cx, cy, cz = sides
    cell = np.repeat(np.arange(cx * cy * cz, dtype=np.int64), k)
    p = rng.random((cell.size, 3), dtype=np.float32).astype(np.float64)
    p[:, 0] += cell % cx
    p[:, 1] += (cell // cx) % cy
    p[:, 2] += cell // (cx * cy)
    if ball:
        p = p[((p - 0.5 * cx) ** 2).sum(1) <= (0.5 * cx) ** 2]
    if len(p) < n:                                     # a small body: fill up at random
        p = np.concatenate([p, p[rng.integers(0, len(p), n - len(p))] * 0.999 + 0.0005 * cx])
    if len(p) > n:
        p = p[np.sort(rng.permutation(len(p))[:n])]
    return p


def _scene(case, seed):
    """Bodies of a scene as (material, x, v) in FP32, in a unit-sized domain."""
    rng = np.random.default_rng([int(seed), 20261202])
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    h = 1.0 / max(nx, ny, nz)
    pad = _pad(nx, ny, nz)
    shapes = _shapes(case["material"], case["n"], case["per_cell"])
    dam = case["material"] == "water"
    width = sum(b[3][0] for b in shapes) + 2.0 * (len(shapes) - 1)
    at = pad + 1.5 if dam else max(pad + 1.5, 0.5 * (nx - width))
    out = []
    for k, (material, n, ball, sides) in enumerate(shapes):
        p = _sample(rng, n, case["per_cell"], ball, sides)
        low = pad + 1.5                                # just above the floor
        side = pad + 1.5 if dam else max(pad + 1.5, 0.5 * (nz - sides[2]))
        p += np.array([at, low, side]) + rng.random(3) * 0.5
        at += sides[0] + 2.0
        x = (p * h).astype(np.float32)
        c = (x.max(0) + x.min(0)).astype(np.float64) / 2
        size = float((x.max(0) - x.min(0)).max())
        d = x.astype(np.float64) - c
        speed, wave, spin = {"jello": ((0.0, -1.0, 0.0), 0.2, 0.3), "snow": ((0.2, 0.0, 0.0), 0.05, 0.6),
                             "water": ((0.3, 0.0, 0.1), 0.3, 0.2)}[material]
        v = np.tile(np.array(speed), (n, 1))
        if material == "snow":
            v[:, 0] *= (12.0 if case["cfl"] else 1.0) * (-1.0 if k == len(shapes) - 1 else 1.0)
        axis = rng.normal(0, 1, 3)
        v += np.cross(axis / np.linalg.norm(axis) * (2 * spin / size), d)      # `spin` m/s at the sides
        for a in range(3):
            turn = rng.normal(0, 1, 3)
            v[:, a] += wave * np.sin(2 * math.pi * (d @ (turn / np.linalg.norm(turn))) / size + rng.random() * 6.28)
        out.append((material, x, v.astype(np.float32)))
    if case["material"] != "mixed":                    # one particle group
        out = [(case["material"], np.concatenate([b[1] for b in out]), np.concatenate([b[2] for b in out]))]
    return out


def _config(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    kw = dict(h=1.0 / max(nx, ny, nz), nx=nx, ny=ny, nz=nz, dt=case["dt"], bc_pad=_pad(nx, ny, nz),
              bc_mode=capi.BC_STICKY if case["material"] == "jello" else capi.BC_AXIS)
    if case["cfl"]:
        kw.update(dt_mode=capi.DT_CFL, cfl=CFL)
    return capi.default_config(**kw)


def _sim(case, seed):
    cfg = _config(case)
    sim = capi.Sim(cfg)
    for material, x, v in _scene(case, seed):
        m = PARAMS[material]
        sim.add_particles(capi.material(m["E"], m["nu"], m["rho"], TYPES[material], **m["extra"]), x, vel=v,
                          volume=cfg.h ** 3)
    return sim


def _batch_scenes(case):
    m = case["scenes"]
    out = []
    for k in range(m):
        n = int(case["n_min"] * (case["n_max"] / case["n_min"]) ** ((k * 7 % m) / max(1, m - 1)))
        material = ("jello", "snow", "water")[k % 3]
        need = max(_extent(material, n, 6.0)) - 14    # 3-cell walls
        grid = min((g for g in BATCH_GRIDS if g >= need), default=256)
        out.append(dict(material=material, n=n, nx=grid, ny=grid, nz=grid, per_cell=6.0, cfl=False,
                        dt=_dt(material, grid)))
    return out


def _squares(case, seed):
    """Three squares of uniform random particles, as the 2D workload stacks
    them, falling and spinning slowly: positions and velocities."""
    rng = np.random.default_rng([int(seed), 2])
    x, v = [], []
    for g, part in enumerate(np.array_split(np.empty(case["n"]), 3)):
        d = rng.random((len(part), 2)) * 0.2
        spin = rng.choice((-1.0, 1.0)) * rng.uniform(4.0, 8.0)
        x.append(d + np.array([0.3 + 0.1 * g, 0.05 + 0.32 * g]))
        v.append(np.array([0.0, -0.5]) + spin * (d - 0.1)[:, ::-1] * np.array([-1.0, 1.0]))
    return np.concatenate(x).astype(np.float32), np.concatenate(v).astype(np.float32)


# ---------------------------------------------------------------------------

def prepare(case, seed):
    if case["kind"] == "scene":
        return dict(case=case, sim=_sim(case, seed))
    if case["kind"] == "batch":
        sims = [_sim(c, seed + 101 * k) for k, c in enumerate(_batch_scenes(case))]
        return dict(case=case, sims=sims, batch=capi.Batch(sims))
    sim = capi.Sim2D(n_grid=case["n_grid"], dt=case["dt"])
    x, v = _squares(case, seed)
    sim.add_particles(x, v)
    return dict(case=case, sim=sim)


def _materials(case):
    return ["jello", "water", "snow"] if case["material"] == "mixed" else [case["material"]]


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        state["batch"].run(case["steps"])
        return [s.read(0, capi.P_POS) for s in state["sims"]]
    sim = state["sim"]
    sim.run(case["steps"])
    if case["kind"] == "snow2d":
        return dict(x=sim.read(capi.P2_POS), v=sim.read(capi.P2_VEL), F=sim.read(capi.P2_F), J=sim.read(capi.P2_JP))
    if case["read"] == "positions":
        return sim.positions()
    if case["read"] == "viewer":
        return dict(x=sim.positions(), v=np.concatenate([sim.read(g, capi.P_VEL) for g in range(sim.group_count())]))
    return [{f: sim.read(g, FIELD[f]) for f in STATE[m]} for g, m in enumerate(_materials(case))]


def work(case):
    """Every step reads and writes each particle's state once and writes and
    reads each node with mass once; a pass hands out what it reads."""
    if case["kind"] == "batch":
        parts = [work(dict(c, kind="scene", steps=case["steps"], read="positions")) for c in _batch_scenes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if case["kind"] == "snow2d":
        n, steps = case["n"], case["steps"]
        nodes = 0.12 * 1.2 * case["n_grid"] ** 2
        return {"bytes": steps * (n * 13 * 8 + nodes * 20) + n * 9 * 8, "flops": steps * n * 450.0}
    total = {"bytes": 0.0, "flops": 0.0}
    for material, n, ball, sides in _shapes(case["material"], case["n"], case["per_cell"]):
        floats = sum(FLOATS[f] for f in STATE[material])
        nodes = 1.15 * n / case["per_cell"]
        read = dict(positions=3, viewer=6, state=floats)[case["read"]]
        total["bytes"] += case["steps"] * (n * floats * 8 + nodes * 28) + n * read * 8
        total["flops"] += case["steps"] * n * (750.0 if material == "water" else 1000.0)
    return total


# ---------------------------------------------------------------------------
# The same passes in 64 bits.

def _weights(f):
    """Quadratic B-spline weights and their derivatives at the three nodes of
    an axis, f in [0.5, 1.5] the distance from the first in cells."""
    return (torch.stack([0.5 * (1.5 - f) ** 2, 0.75 - (f - 1) ** 2, 0.5 * (f - 0.5) ** 2]),
            torch.stack([f - 1.5, -2 * (f - 1), f - 0.5]))


def _cofactor(R):
    a, b, c = R[:, 0], R[:, 1], R[:, 2]
    return torch.stack([torch.linalg.cross(b, c), torch.linalg.cross(c, a), torch.linalg.cross(a, b)], 1)


def _mul(A, B):
    return (A[:, :, :, None] * B[:, None, :, :]).sum(2)


def _polar(F):
    R = F
    for _ in range(7):
        c = _cofactor(R)
        R = 0.5 * (R + c / (R[:, 0] * c[:, 0]).sum(1)[:, None, None])
    return R


def _jacobi(S):
    """Eigenvalues and eigenvectors (columns) of symmetric 3x3 matrices."""
    S = S.clone()
    V = torch.eye(3, dtype=S.dtype, device=S.device).repeat(len(S), 1, 1)
    for _ in range(6):
        for p, q in ((0, 1), (0, 2), (1, 2)):
            th = 0.5 * torch.atan2(2 * S[:, p, q], S[:, q, q] - S[:, p, p])
            c, s = torch.cos(th)[:, None], torch.sin(th)[:, None]
            for M in (S, V):
                a, b = M[:, :, p].clone(), M[:, :, q].clone()
                M[:, :, p], M[:, :, q] = c * a - s * b, s * a + c * b
            a, b = S[:, p].clone(), S[:, q].clone()
            S[:, p], S[:, q] = c * a - s * b, s * a + c * b
    return S.diagonal(dim1=1, dim2=2), V


def _stress(g):
    """Kirchhoff stress of a group: fixed-corotated (snow hardened by J_p) or
    water's pressure."""
    m = g["m"]
    eye = torch.eye(3, dtype=torch.float64, device=g["x"].device)
    if g["material"] == "water":
        J = g["J"][:, 0]
        p = m["extra"]["eos_k"] * (J ** -m["extra"]["eos_gamma"] - 1)
        return (-p * J)[:, None, None] * eye
    mu = m["E"] / (2 * (1 + m["nu"]))
    lam = m["E"] * m["nu"] / ((1 + m["nu"]) * (1 - 2 * m["nu"]))
    F = g["F"]
    J = (F[:, 0] * _cofactor(F)[:, 0]).sum(1)
    hard = torch.exp(m["extra"]["xi"] * (1 - g["J"][:, 0])) if g["material"] == "snow" else torch.ones_like(J)
    return hard[:, None, None] * (2 * mu * _mul(F - _polar(F), F.transpose(1, 2)) +
                                  (lam * J * (J - 1))[:, None, None] * eye)


def _speed(g):
    """The controller's measure: |v| + elastic wave speed."""
    m = g["m"]
    lam = m["E"] * m["nu"] / ((1 + m["nu"]) * (1 - 2 * m["nu"]))
    c2 = (lam + m["E"] / (1 + m["nu"])) / m["rho"] * torch.ones_like(g["J"][:, 0])
    if g["material"] == "snow":
        c2 = c2 * torch.exp(m["extra"]["xi"] * (1 - g["J"][:, 0]))
    return float((g["v"].norm(dim=1) + c2.sqrt()).max())


def _stencil(g, shape, inv_h):
    b = torch.clamp(torch.floor(g["x"] * inv_h - 0.5), min=0)
    b = torch.minimum(b, torch.tensor([s - 3.0 for s in shape], dtype=b.dtype, device=b.device))
    f = g["x"] * inv_h - b
    N, D = zip(*(_weights(f[:, a]) for a in range(3)))
    b = b.to(torch.int64)
    first = (b[:, 2] * shape[1] + b[:, 1]) * shape[0] + b[:, 0]
    for ox in range(3):
        for oy in range(3):
            for oz in range(3):
                w = N[0][ox] * N[1][oy] * N[2][oz]
                dw = torch.stack([D[0][ox] * N[1][oy] * N[2][oz], N[0][ox] * D[1][oy] * N[2][oz],
                                  N[0][ox] * N[1][oy] * D[2][oz]], 1) * inv_h
                o = torch.tensor([ox, oy, oz], dtype=f.dtype, device=f.device)
                yield first + (oz * shape[1] + oy) * shape[0] + ox, w[:, None], dw, (o - f) / inv_h


def _step(groups, shape, h, dt, pad, sticky):
    dev = groups[0]["x"].device
    vol = h ** 3
    grid = torch.zeros((shape[0] * shape[1] * shape[2], 4), dtype=torch.float64, device=dev)
    for g in groups:
        mass = g["m"]["rho"] * vol
        G = -dt * vol * _stress(g)
        for node, w, dw, d in _stencil(g, shape, 1 / h):
            p = mass * w * (g["v"] + (g["C"] * d[:, None, :]).sum(2)) + (G * dw[:, None, :]).sum(2)
            grid.index_add_(0, node, torch.cat([mass * w, p], 1))
    full = grid[:, :1] > 2.220446049250313e-16
    vel = torch.where(full, grid[:, 1:] / torch.where(full, grid[:, :1], 1.0), 0.0)
    vel[:, 1] += -9.8 * dt * full[:, 0]
    vel = vel.reshape(shape[2], shape[1], shape[0], 3)
    for a, dim in ((0, 2), (1, 1), (2, 0)):
        i = torch.arange(shape[a], device=dev)
        wall = torch.nonzero((i <= pad) | (i >= shape[a] - pad))[:, 0]
        sl = [slice(None)] * 3
        sl[dim] = wall
        if sticky:
            vel[tuple(sl)] = 0.0
        else:
            vel[tuple(sl) + (a,)] = 0.0
    vel = vel.reshape(-1, 3)
    for g in groups:
        v = torch.zeros_like(g["v"])
        B = torch.zeros_like(g["C"])
        L = torch.zeros_like(g["C"])
        for node, w, dw, d in _stencil(g, shape, 1 / h):
            u = vel[node]
            v += w * u
            B += (w * u)[:, :, None] * d[:, None, :]
            L += u[:, :, None] * dw[:, None, :]
        g["v"], g["C"] = v, L if g["material"] == "water" else B * (4 / h ** 2)
        if g["material"] == "water":
            g["J"] = g["J"] * (1 + dt * L.diagonal(dim1=1, dim2=2).sum(1))[:, None]
        else:
            g["F"] = g["F"] + dt * _mul(L, g["F"])
        if g["material"] == "snow":
            ev, V = _jacobi(_mul(g["F"].transpose(1, 2), g["F"]))
            s = ev.sqrt()
            ratio = torch.clamp(s, 1 - g["m"]["extra"]["theta_c"], 1 + g["m"]["extra"]["theta_s"]) / s
            clamped = (ratio != 1).any(1)
            Fc = _mul(_mul(g["F"], V) * ratio[:, None, :], V.transpose(1, 2))
            g["F"] = torch.where(clamped[:, None, None], Fc, g["F"])
            g["J"] = g["J"] / ratio.prod(1)[:, None]
        g["x"] = g["x"] + dt * v


def _exact_scene(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    groups = []
    for material, x, v in _scene(case, seed):
        n = len(x)
        groups.append(dict(material=material, m=PARAMS[material],
                           x=torch.from_numpy(x).to(dev, torch.float64), v=torch.from_numpy(v).to(dev, torch.float64),
                           C=torch.zeros((n, 3, 3), dtype=torch.float64, device=dev),
                           F=torch.eye(3, dtype=torch.float64, device=dev).repeat(n, 1, 1),
                           J=torch.ones((n, 1), dtype=torch.float64, device=dev)))
    shape = (case["nx"], case["ny"], case["nz"])
    h = 1.0 / max(shape)
    for _ in range(case["steps"]):
        dt = min([case["dt"]] + [CFL * h / _speed(g) for g in groups if case["cfl"]])
        _step(groups, shape, h, dt, _pad(*shape), case["material"] == "jello")
    return groups


def _exact_2d(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x, v = (torch.from_numpy(a).to(dev, torch.float64) for a in _squares(case, seed))
    n, N, dt = len(x), case["n_grid"], case["dt"]
    dx = 1.0 / N
    vol = 0.25 * dx * dx
    mu0, lam0 = 1e3 / 2.4, 1e3 * 0.2 / (1.2 * 0.6)
    C = torch.zeros((n, 2, 2), dtype=x.dtype, device=dev)
    F = torch.eye(2, dtype=x.dtype, device=dev).repeat(n, 1, 1)
    J = torch.ones(n, dtype=x.dtype, device=dev)
    eye = torch.eye(2, dtype=x.dtype, device=dev)
    i = torch.arange(N, device=dev)
    wall = (i <= 5) | (i >= N - 5)
    wall = (wall[:, None] | wall[None, :]).reshape(-1)

    def nodes():
        b = (x * N - 0.5).to(torch.int64)
        f = x * N - b
        W = [_weights(f[:, a]) for a in range(2)]
        for a in range(3):
            for c in range(3):
                w = W[0][0][a] * W[1][0][c]
                dw = torch.stack([W[0][1][a] * W[1][0][c], W[0][0][a] * W[1][1][c]], 1) * N
                d = torch.stack([a - f[:, 0], c - f[:, 1]], 1) * dx
                yield (b[:, 1] + c) * N + b[:, 0] + a, w[:, None], dw, d

    def polar(M):
        co, si = M[:, 0, 0] + M[:, 1, 1], M[:, 1, 0] - M[:, 0, 1]
        r = torch.hypot(co, si)
        return torch.stack([torch.stack([co / r, -si / r], 1), torch.stack([si / r, co / r], 1)], 1)

    for _ in range(case["steps"]):
        hard = torch.exp(10.0 * (1 - J))
        det = F[:, 0, 0] * F[:, 1, 1] - F[:, 0, 1] * F[:, 1, 0]
        tau = ((2 * mu0 * hard)[:, None, None] * _mul(F - polar(F), F.transpose(1, 2)) +
               (hard * lam0 * (det - 1) * det)[:, None, None] * eye)
        grid = torch.zeros((N * N, 3), dtype=x.dtype, device=dev)
        for node, w, dw, d in nodes():
            p = vol * w * (v + (C * d[:, None, :]).sum(2)) - dt * vol * (tau * dw[:, None, :]).sum(2)
            grid.index_add_(0, node, torch.cat([vol * w, p], 1))
        full = grid[:, :1] > 0
        u = torch.where(full, grid[:, 1:] / torch.where(full, grid[:, :1], 1.0), 0.0)
        u[:, 1] += -50.0 * dt * full[:, 0]
        u[wall] = 0.0
        v, C, L = torch.zeros_like(v), torch.zeros_like(C), torch.zeros_like(C)
        for node, w, dw, d in nodes():
            un = u[node]
            v = v + w * un
            C = C + (4 / dx ** 2) * (w * un)[:, :, None] * d[:, None, :]
            L = L + un[:, :, None] * dw[:, None, :]
        F = F + dt * _mul(L, F)
        S = _mul(F.transpose(1, 2), F)
        th = 0.5 * torch.atan2(2 * S[:, 0, 1], S[:, 0, 0] - S[:, 1, 1])
        co, si = torch.cos(th), torch.sin(th)
        V = torch.stack([torch.stack([co, -si], 1), torch.stack([si, co], 1)], 1)
        FV = _mul(F, V)
        s = FV.norm(dim=1)
        ratio = torch.clamp(s, 1 - 2.5e-2, 1 + 7.5e-3) / s
        F = torch.where((ratio != 1).any(1)[:, None, None], _mul(FV * ratio[:, None, :], V.transpose(1, 2)), F)
        J = J / ratio.prod(1)
        x = x + dt * v
    return dict(x=x, v=v, F=F.reshape(n, 4), J=J[:, None])


def exact(case, seed):
    if case["kind"] == "snow2d":
        return _exact_2d(case, seed)
    if case["kind"] == "batch":
        return [_exact_scene(dict(c, steps=case["steps"]), seed + 101 * k)[0]["x"]
                for k, c in enumerate(_batch_scenes(case))]
    groups = _exact_scene(case, seed)
    if case["read"] == "positions":
        return torch.cat([g["x"] for g in groups])
    if case["read"] == "viewer":
        return dict(x=torch.cat([g["x"] for g in groups]), v=torch.cat([g["v"] for g in groups]))
    return [{f: g[f].reshape(len(g["x"]), -1) for f in STATE[g["material"]]} for g in groups]
