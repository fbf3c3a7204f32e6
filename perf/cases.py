"""Performance cases of the uniform-MAC step: what users of the library run, from single projections of a few
thousand cells to full steps of the largest grids, through the public entry points of fluidsim_amd.

Every pass starts from a device-resident snapshot (a run that is restarted, a served request, a parameter sweep),
runs one solve, a few steps or a batch, and reads the fields back into page-locked host arrays that the program
keeps, as a caller of fs_download does.  Sizes and settings are those of the repository's benchmark and tests (the
128^2 dam break, the 1024^2 vortex box, the 2048^2 obstacle tank, the 64..512 batch, the 128..2048 request
stream, 1920 x 1080 and 512 x 420 scenes), plus odd and thin grids.
"""
import ctypes
import math

import numpy as np
import torch

import fluidsim_amd as F
from fluidsim_amd import _abi
from fluidsim_amd import workloads as WL

RB, CHEB = F.FS_SMOOTHER_RED_BLACK, F.FS_SMOOTHER_CHEBYSHEV
PRECISION = {"fp32": F.FS_MG_FP32, "fp16": F.FS_MG_FP16, "bf16": F.FS_MG_BF16}


def listed():
    return [
        # The smallest interactive grid: one pressure solve whose whole multigrid hierarchy is one workgroup's
        # work; launches and the coarse end are all there is.
        dict(name="project_61x47", kind="project", scene="pool", w=61, h=47, smoother="red_black", sweeps=4,
             coarse=4, precision="fp32"),
        # The reference test suite's odd grid (two-phase pool), with the reference's own V(4,4) red-black cycle.
        dict(name="project_513x257", kind="project", scene="pool", w=513, h=257, smoother="red_black", sweeps=4,
             coarse=4, precision="fp32"),
        # The headline benchmark: a projection of the 1024^2 vortex box with the smoother its tuner selects.
        dict(name="project_1024", kind="project", scene="vortex", w=1024, h=1024, smoother="chebyshev", sweeps=3,
             coarse=2, precision="fp32"),
        # The hardest solve: free surface (1000:1) and obstacles at 2048^2, tuned smoother.  The largest case.
        dict(name="tank_2048", kind="project", scene="tank", w=2048, h=2048, smoother="chebyshev", sweeps=8,
             coarse=4, precision="fp32"),
        # The same on a ragged grid with the reference's cycle and bfloat16 multigrid levels.
        dict(name="tank_1000x700_bf16", kind="project", scene="tank", w=1000, h=700, smoother="red_black", sweeps=4,
             coarse=4, precision="bf16"),
        # A small full simulation at the defaults: PLIC transport, gravity and projection of a 128^2 dam break.
        dict(name="dam_break_128", kind="step", scene="dam", w=128, h=128, steps=4, liquids=1, gases=1,
             viscous=False, tension=False, smoother="red_black", sweeps=4, coarse=4, vis_sweeps=0),
        # A full-HD two-phase pool of two liquids and two gases (the reference's timing table), defaults.
        dict(name="step_1920x1080", kind="step", scene="pool", w=1920, h=1080, steps=2, liquids=2, gases=2,
             viscous=False, tension=False, smoother="red_black", sweeps=4, coarse=4, vis_sweeps=0),
        # A request of the serving stream: transport, viscosity, surface tension, projection, served smoothers.
        dict(name="request_1594x837", kind="step", scene="pool", w=1594, h=837, steps=2, liquids=1, gases=1,
             viscous=True, tension=True, smoother="chebyshev", sweeps=8, coarse=3, vis_sweeps=4),
        # Smoke-like flow: semi-Lagrangian steps of the 1024^2 vortex box (advection, gravity, projection).
        dict(name="semi_lagrangian_1024", kind="smoke", w=1024, h=1024, steps=8),
        # Transport alone: four-ingredient PLIC/VOF advection, as a caller coupling its own forces runs it.
        dict(name="advect_700x500", kind="advect", w=700, h=500, steps=10, liquids=2, gases=2),
        # The viscosity solve on the caller's own device arrays, without allocation.
        dict(name="viscosity_641x363", kind="viscosity", w=641, h=363, nu=0.1),
        # A parameter sweep: many small grids with obstacles projected in one batch.
        dict(name="batch_32", kind="batch", count=32, low=64, high=512, split=131072),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _smoother(rng):
    if rng.random() < 0.5:
        return dict(smoother="red_black", sweeps=rng.choice([3, 4]), coarse=4)
    return dict(smoother="chebyshev", sweeps=rng.choice([3, 4, 5, 6, 8]), coarse=rng.choice([3, 4]))


def draw(rng):
    kind = rng.choice(["pool", "vortex", "tank", "tank16", "dam", "scene", "request", "smoke", "advect", "viscosity",
                       "batch"])
    if kind == "pool":
        return dict(kind="project", scene="pool", w=_log_int(rng, 24, 1200), h=_log_int(rng, 24, 1200),
                    precision="fp32", **_smoother(rng))
    if kind == "vortex":
        return dict(kind="project", scene="vortex", w=_log_int(rng, 96, 2048), h=_log_int(rng, 96, 2048),
                    precision="fp32", **_smoother(rng))
    if kind == "tank":
        return dict(kind="project", scene="tank", w=_log_int(rng, 160, 1600), h=_log_int(rng, 160, 1600),
                    precision="fp32", **_smoother(rng))
    if kind == "tank16":
        return dict(kind="project", scene="tank", w=_log_int(rng, 160, 1000), h=_log_int(rng, 160, 1000),
                    smoother="red_black", sweeps=4, coarse=4, precision=rng.choice(["fp16", "bf16"]))
    if kind == "dam":
        return dict(kind="step", scene="dam", w=_log_int(rng, 40, 256), h=_log_int(rng, 40, 256),
                    steps=rng.randint(2, 4), liquids=1, gases=1, viscous=False, tension=False, smoother="red_black",
                    sweeps=4, coarse=4, vis_sweeps=0)
    if kind == "scene":
        return dict(kind="step", scene="pool", w=_log_int(rng, 200, 1920), h=_log_int(rng, 200, 1080),
                    steps=2, liquids=rng.randint(1, 2), gases=rng.randint(1, 2), viscous=False, tension=False,
                    smoother="red_black", sweeps=4, coarse=4, vis_sweeps=0)
    if kind == "request":
        return dict(kind="step", scene="pool", w=_log_int(rng, 128, 1400), h=_log_int(rng, 128, 1400), steps=2,
                    liquids=1, gases=1, viscous=True, tension=True, vis_sweeps=rng.choice([0, 2, 4, 6]),
                    **_smoother(rng))
    if kind == "smoke":
        return dict(kind="smoke", w=_log_int(rng, 96, 1400), h=_log_int(rng, 96, 1400), steps=rng.randint(4, 8))
    if kind == "advect":
        return dict(kind="advect", w=_log_int(rng, 100, 1200), h=_log_int(rng, 100, 1200), steps=rng.randint(4, 10),
                    liquids=rng.randint(1, 2), gases=rng.randint(1, 2))
    if kind == "viscosity":
        return dict(kind="viscosity", w=_log_int(rng, 33, 700), h=_log_int(rng, 33, 700),
                    nu=math.exp(rng.uniform(math.log(1e-3), math.log(0.5))))
    return dict(kind="batch", count=rng.randint(6, 32), low=64, high=rng.randint(200, 512),
                split=rng.choice([0, 131072]))


# ---- inputs ----

def _flow(rng, w, h, cell, vortices, sources, low, high, scale):
    """Gaussian vortices and divergent sources (the benchmark's law), as sums of outer products."""
    n = vortices + sources
    cx, cy = rng.uniform(n, 0.0, w * cell), rng.uniform(n, 0.0, h * cell)
    radius, strength = rng.uniform(n, low, high), rng.normal(n) * scale

    def parts(x, y):
        dx, dy = x[None, :] * cell - cx[:, None], y[:, None] * cell - cy[None, :]
        return dx, dy, np.exp(-dx * dx / (2.0 * radius[:, None] ** 2)), np.exp(-dy * dy / (2.0 * radius ** 2)) * strength

    k = vortices
    dx, dy, ex, ey = parts(np.arange(w + 1.0), np.arange(h) + 0.5)
    u = -(dy * ey)[:, :k] @ ex[:k] + ey[:, k:] @ (dx * ex)[k:]
    dx, dy, ex, ey = parts(np.arange(w) + 0.5, np.arange(h + 1.0))
    v = ey[:, :k] @ (dx * ex)[:k] + (dy * ey)[:, k:] @ ex[k:]
    u, v = u.ravel(), v.ravel()
    WL.zero_walls(u, v, w, h)
    return u, v


def _split(mass, parts, w, h, rng):
    """A mass field as `parts` ingredients in smoothly varying proportions."""
    if parts == 1:
        return mass
    a, b, c = rng.uniform(3, 0.5, 3.0)
    x, y = np.arange(w)[None, :] / w * math.pi, np.arange(h)[:, None] / h * math.pi
    share = 0.5 + 0.4 * np.sin(a * x + b) * np.cos(c * y)
    first = mass * share.ravel()
    return np.concatenate([first, mass - first])


def _pool(case, seed, scale=1.0):
    """A pool with a drop above it and random vortices: a 1000:1 free surface in a closed box."""
    w, h, rng = case["w"], case["h"], WL.SplitMix64(seed)
    cell = 1.0 / max(w, h)
    fraction = WL.pool_with_drop(w, h, cell, rng.uniform(1, 0.3, 0.9)[0], 0.08, rng)
    u, v = _flow(rng, w, h, cell, 8, 0, 0.02, 0.08, scale)
    liquid, gas = WL.two_phase_masses(fraction, cell)
    liquids, gases = case.get("liquids", 1), case.get("gases", 1)
    return WL.Workload("pool", w, h, cell, [100.0] * liquids, [0.1] * gases, 9.81, 1.0 / 240.0, fraction, u, v,
                       _split(liquid, liquids, w, h, rng), _split(gas, gases, w, h, rng), {"seed": seed, "solid": None})


def _box(case, seed, tank):
    """The vortex box (64 vortices, 16 sources, one liquid), or as a tank: 42 circles and boxes over about 15% of
    the cells, one in each field of a 7 x 6 raster so that the fluid stays connected, and air in the top 30%."""
    w, h, rng = case["w"], case["h"], WL.SplitMix64(seed)
    cell = 1.0 / max(w, h)
    u, v = _flow(rng, w, h, cell, 64, 16, 0.01, 0.05, 1.0)
    fraction, solid = np.ones((h, w)), None
    if tank:
        px, py = w / 7.0, h / 6.0
        size = rng.uniform(42, 0.14, 0.28)
        x = (np.arange(42) % 7 + rng.uniform(42, 0.3, 0.7)) * px
        y = (np.arange(42) // 7 + rng.uniform(42, 0.3, 0.7)) * py
        solid = np.zeros((h, w), dtype=np.uint8)
        for k in range(42):
            dx, dy = np.abs(np.arange(w) + 0.5 - x[k]) / px, np.abs(np.arange(h) + 0.5 - y[k]) / py
            xs, ys = np.flatnonzero(dx < size[k]), np.flatnonzero(dy < size[k])
            if xs.size and ys.size:
                inside = np.hypot(dx[xs][None, :], dy[ys][:, None]) < size[k]
                solid[ys[0]:ys[-1] + 1, xs[0]:xs[-1] + 1] |= (inside | (k % 2 == 1)).astype(np.uint8)
        fraction[:int(0.3 * h)] = 0.0
        fraction[solid != 0] = 0.0
        solid = solid.ravel()
    fraction = fraction.ravel()
    liquid, gas = WL.two_phase_masses(fraction, cell)
    return WL.Workload("box", w, h, cell, [100.0], [0.1], 9.81, 1.0 / 120.0, fraction, u, v, liquid, gas,
                       {"seed": seed, "solid": solid})


def _instances(case, seed):
    """The grids of a batch: sides log-uniform in [low, high] (the same for every seed), pools with a drop, vortices
    and, in three of four, the tank's obstacles in smaller number."""
    sides = WL.SplitMix64(1009 * case["count"] + case["high"])
    out = []
    for k in range(case["count"]):
        w, h = (int(round(math.exp(x))) for x in sides.uniform(2, math.log(case["low"]), math.log(case["high"])))
        wl = _pool(dict(w=w, h=h), 1000003 * seed + k)
        if k % 4:
            solid = _box(dict(w=w, h=h), 1000003 * seed + k, True).meta["solid"]
            wl.fraction[solid != 0] = 0.0
            wl.liquid_mass, wl.gas_mass = WL.two_phase_masses(wl.fraction, wl.cell_size)
            wl.meta["solid"] = solid
        out.append(wl)
    return out


def _workload(case, seed):
    scene = case.get("scene", "vortex")
    if scene == "dam":
        return WL.dam_break(case["w"], case["h"], seed)
    if scene == "pool":
        return _pool(case, seed, scale=0.05 if case.get("viscous") else 1.0)
    return _box(case, seed, scene == "tank")


def _grid(wl, context=None):
    grid = F.FluidGridHIP(wl.width, wl.height, wl.cell_size, context)
    WL.load_into(grid, wl)
    if wl.meta.get("solid") is not None:
        grid.setSolidMask(wl.meta["solid"])
    grid.setRelativeTolerance(True)
    return grid


def _host(n):
    return torch.empty(n, dtype=torch.float64, pin_memory=torch.cuda.is_available())


class _Fields:
    """The program's page-locked host arrays and the read-back of a grid's fields into them."""

    def __init__(self, wl, names):
        n = wl.width * wl.height
        sizes = dict(f=n, u=(wl.width + 1) * wl.height, v=wl.width * (wl.height + 1), p=n,
                     liquid=n * len(wl.liquid_density), gas=n * len(wl.gas_density))
        self.host = {k: _host(sizes[k]) for k in names}
        self.pointers = [ctypes.cast(self.host[k].data_ptr(), ctypes.POINTER(ctypes.c_double)) if k in names else None
                         for k in ("f", "u", "v", "p", "liquid", "gas")]

    def read(self, grid):
        _abi.call("fs_download", grid.handle, *self.pointers)
        return self.host


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        context = F.Context(0)
        context.set_batch_split(case["split"])
        loads = _instances(case, seed)
        grids = [_grid(wl, context) for wl in loads]
        for grid in grids:
            grid.snapshotSave()
        sizes = [(wl.width, wl.height) for wl in loads]
        host = {"u": _host(sum((w + 1) * h for w, h in sizes)), "v": _host(sum(w * (h + 1) for w, h in sizes))}
        pointers, at = [], {"u": 0, "v": 0}
        for w, h in sizes:
            row = []
            for name, n in (("u", (w + 1) * h), ("v", w * (h + 1))):
                row.append(ctypes.cast(host[name].data_ptr() + 8 * at[name], ctypes.POINTER(ctypes.c_double)))
                at[name] += n
            pointers.append(row)
        return dict(kind=kind, context=context, grids=grids, host=host, pointers=pointers, dt=1.0 / 240.0)
    if kind == "viscosity":
        w, h, rng = case["w"], case["h"], WL.SplitMix64(seed)
        wl = _pool(case, seed)
        mixture = np.stack([100.0 * wl.fraction + 0.1 * (1.0 - wl.fraction), np.zeros(w * h)], axis=1)
        mixture[:, 1] = case["nu"] * mixture[:, 0] * (0.5 + rng.uniform(w * h))
        u, v = (a + 0.2 * WL.SplitMix64(seed + k).normal(a.size) for k, a in ((1, wl.u), (2, wl.v)))
        WL.zero_walls(u, v, w, h)
        put = [torch.from_numpy(np.ascontiguousarray(a).ravel()).cuda() for a in (mixture, u, v)]
        torch.cuda.synchronize()
        return dict(kind=kind, w=w, h=h, cell=wl.cell_size, material=put[0], u0=put[1], v0=put[2],
                    u=torch.empty_like(put[1]), v=torch.empty_like(put[2]), context=F.default_context(), dt=1e-3)
    wl = _workload(case, seed) if kind != "advect" else _pool(case, seed)
    grid = _grid(wl)
    state = dict(kind=kind, grid=grid, dt=wl.dt, steps=case.get("steps", 1))
    if kind == "project":
        grid.setPressureSmoother(CHEB if case["smoother"] == "chebyshev" else RB, case["sweeps"], case["coarse"])
        grid.setMultigridPrecision(PRECISION[case["precision"]])
        # with obstacles the velocity is the result: the pressure inside solid cells has no meaning
        state["fields"] = _Fields(wl, ("u", "v") if case["scene"] == "tank" else ("u", "v", "p"))
    elif kind == "step":
        grid.setPressureSmoother(CHEB if case["smoother"] == "chebyshev" else RB, case["sweeps"], case["coarse"])
        if case["viscous"]:
            nu = 0.05
            for k in range(case["liquids"]):
                grid.setComponentViscosity("liquid", k, nu * 100.0)
            for k in range(case["gases"]):
                grid.setComponentViscosity("gas", k, nu * 0.1)
            grid.setViscositySmoother(case["vis_sweeps"])
        if case["tension"]:
            grid.setSurfaceTension(0.04)
            state["dt"] = 0.5 * grid.capillaryStepLimit()
        state["fields"] = _Fields(wl, ("f", "u", "v", "p", "liquid", "gas"))
    elif kind == "smoke":
        grid.setTransport(F.FS_TRANSPORT_SEMI_LAGRANGIAN)
        grid.setPressureSmoother(CHEB, 3, 2)
        state["fields"] = _Fields(wl, ("u", "v", "p"))
    else:
        state["dt"] = 0.5 * wl.cell_size / max(np.abs(wl.u).max(), np.abs(wl.v).max(), 1e-3)
        state["fields"] = _Fields(wl, ("f", "u", "v", "liquid", "gas"))
    grid.snapshotSave()
    return state


def run(state):
    kind = state["kind"]
    if kind == "batch":
        for grid in state["grids"]:
            grid.snapshotRestore()
        F.batch_project(state["grids"], state["dt"], 2000, 1e-6)
        for grid, (u, v) in zip(state["grids"], state["pointers"]):
            _abi.call("fs_download", grid.handle, None, u, v, None, None, None)
        return state["host"]
    if kind == "viscosity":
        state["u"].copy_(state["u0"])
        state["v"].copy_(state["v0"])
        torch.cuda.current_stream().synchronize()   # the library's stream reads the arrays
        done, relative = ctypes.c_int(), ctypes.c_double()
        _abi.call("fs_viscosity_solve_noalloc", state["context"].handle, state["w"], state["h"], state["cell"],
                  *(ctypes.cast(state[k].data_ptr(), ctypes.POINTER(ctypes.c_double)) for k in ("material", "u", "v")),
                  state["dt"], 1e-4, -1, ctypes.byref(done), ctypes.byref(relative))
        return {"u": state["u"], "v": state["v"]}
    grid = state["grid"]
    grid.snapshotRestore()
    if kind == "project":
        grid.project(state["dt"], 2000, 1e-6)
    elif kind == "advect":
        for _ in range(state["steps"]):
            grid.advect(state["dt"])
    else:
        for _ in range(state["steps"]):
            grid.step(state["dt"], 2000, 1e-6)
    return state["fields"].read(grid)


# ---- what a pass cannot do without ----

def work(case):
    """Bytes: each input field read once and each result written once, per solve or step.  Operations: of one
    multigrid-preconditioned pass over the unknowns per solve or step (the iteration count is the solver's)."""
    kind = case["kind"]
    if kind == "batch":
        n = case["count"] * (0.5 * (case["low"] + case["high"])) ** 2 * 0.6
        return dict(bytes=n * 8 * (2 + 2 + 2), flops=n * 150.0)
    n = float(case["w"] * case["h"])
    fields = 1 + case.get("liquids", 1) + case.get("gases", 1)
    steps = case.get("steps", 1)
    if kind == "project":   # masses, u, v read; u, v, p written
        return dict(bytes=n * 8 * (2 + 2 + 3), flops=n * 150.0)
    if kind == "viscosity":   # material, u, v read; u, v written
        return dict(bytes=n * 8 * (2 + 2 + 2), flops=n * 250.0)
    if kind == "advect":   # fraction, masses, u, v read and written
        return dict(bytes=steps * n * 16 * (fields + 2), flops=steps * n * 300.0)
    extra = 400.0 if case.get("viscous") else 0.0
    return dict(bytes=steps * n * 16 * (fields + 3), flops=steps * n * (450.0 + extra))


def tolerance(case):
    kind = case["kind"]
    if kind == "advect":
        return "exact"   # the transport evaluates the reference's FP64 expressions in the reference's order
    if kind == "viscosity" or case.get("viscous"):
        # the viscosity solve stops at a relative residual of 1e-4, looked at every four iterations: measured 2e-4 to
        # 1e-3 from the 64-bit solution (the largest face difference 0.03 of the RMS), 7e-4 and 0.06 between smoothers
        return {"rel": 1e-3, "max": 1e-1}
    # pressure solves stop at a relative residual of 1e-6: measured at most 5.6e-7 (largest 2.1e-5) between solves of
    # the same input with other smoothers, and 5.5e-7 from the 64-bit solution
    return {"rel": 2e-6, "max": 1e-4}


# ---- the same in 64 bits, in plain torch ----

def _project64(u, v, density, solid, cell, dt):
    """The projection of (u, v), h x (w + 1) and (h + 1) x w: closed walls, faces of solid cells closed, weights
    2 / (rho_a + rho_b); diagonally preconditioned CG to 1e-11 of max|b|.  Returns u, v, p."""
    h, w = density.shape
    wx = torch.zeros_like(u)
    wy = torch.zeros_like(v)
    wx[:, 1:w] = 2.0 / (density[:, 1:] + density[:, :-1])
    wy[1:h] = 2.0 / (density[1:] + density[:-1])
    if solid is not None:
        wx[:, 1:w][solid[:, 1:] | solid[:, :-1]] = 0.0
        wy[1:h][solid[1:] | solid[:-1]] = 0.0
    u, v = torch.where(wx > 0, u, 0.0), torch.where(wy > 0, v, 0.0)
    b = -((u[:, 1:] - u[:, :-1]) + (v[1:] - v[:-1])) / cell * (cell * cell / dt)
    fluid = torch.ones_like(b) if solid is None else (~solid).double()
    b = (b - (b * fluid).sum() / fluid.sum()) * fluid
    diagonal = wx[:, 1:] + wx[:, :-1] + wy[1:] + wy[:-1]
    inverse = torch.where(diagonal > 0, 1.0 / diagonal, 0.0)
    fx, fy = torch.zeros_like(u), torch.zeros_like(v)

    def apply(p):
        torch.sub(p[:, 1:], p[:, :-1], out=fx[:, 1:w])
        torch.sub(p[1:], p[:-1], out=fy[1:h])
        fx.mul_(wx)
        fy.mul_(wy)
        return (fx[:, :-1] - fx[:, 1:]).add_(fy[:-1]).sub_(fy[1:])

    p, r = torch.zeros_like(b), b.clone()
    z = r * inverse
    d = z.clone()
    rz = (r * z).sum()
    goal = 1e-11 * float(b.abs().max())
    for k in range(40000):
        if k % 200 == 0 and float(r.abs().max()) <= goal:
            break
        q = apply(d)
        alpha = rz / (d * q).sum()
        p.addcmul_(d, alpha)
        r.addcmul_(q, -alpha)
        torch.mul(r, inverse, out=z)
        rz, last = (r * z).sum(), rz
        d.mul_(rz / last).add_(z)
    p = (p - (p * fluid).sum() / fluid.sum()) * fluid
    u[:, 1:w] -= (p[:, 1:] - p[:, :-1]) / cell * dt * wx[:, 1:w]
    v[1:h] -= (p[1:] - p[:-1]) / cell * dt * wy[1:h]
    return u, v, p


def _poisson64(u, v, density, cell, dt):
    """The projection for one constant density: the Neumann problem is diagonal in cosines."""
    h, w = u.shape[0], v.shape[1]
    u, v = u.clone(), v.clone()
    u[:, 0] = u[:, w] = 0.0
    v[0] = v[h] = 0.0
    b = -((u[:, 1:] - u[:, :-1]) + (v[1:] - v[:-1])) / cell * (cell * cell / dt)
    even = torch.cat([torch.cat([b, b.flip(1)], 1), torch.cat([b, b.flip(1)], 1).flip(0)], 0)
    kx = torch.arange(2 * w, device=b.device, dtype=torch.float64) * (math.pi / w)
    ky = torch.arange(2 * h, device=b.device, dtype=torch.float64) * (math.pi / h)
    symbol = (4.0 - 2.0 * torch.cos(kx)[None, :] - 2.0 * torch.cos(ky)[:, None]) / density
    symbol[0, 0] = 1.0
    spectrum = torch.fft.fft2(even) / symbol
    spectrum[0, 0] = 0.0
    p = torch.fft.ifft2(spectrum).real[:h, :w].contiguous()
    p -= p.mean()
    u[:, 1:w] -= (p[:, 1:] - p[:, :-1]) / cell * dt / density
    v[1:h] -= (p[1:] - p[:-1]) / cell * dt / density
    return u, v, p


def _sample64(field, x, y):
    h, w = field.shape
    x, y = x.clamp(0.0, w - 1.0), y.clamp(0.0, h - 1.0)
    x0, y0 = x.long(), y.long()
    x1, y1 = (x0 + 1).clamp(max=w - 1), (y0 + 1).clamp(max=h - 1)
    tx, ty = x - x0, y - y0
    top = (1.0 - tx) * field[y0, x0] + tx * field[y0, x1]
    low = (1.0 - tx) * field[y1, x0] + tx * field[y1, x1]
    return (1.0 - ty) * top + ty * low


def _smoke64(wl, steps):
    """Semi-Lagrangian steps of a one-density box: midpoint backtraces, gravity, projection (in cells)."""
    w, h, cell, dt = wl.width, wl.height, wl.cell_size, wl.dt
    u, v = (torch.from_numpy(a).cuda() for a in (wl.u.reshape(h, w + 1), wl.v.reshape(h + 1, w)))

    def back(x, y):   # positions in cells
        vx, vy = _sample64(u, x, y - 0.5), _sample64(v, x - 0.5, y)
        mx, my = x - 0.5 * dt / cell * vx, y - 0.5 * dt / cell * vy
        vx, vy = _sample64(u, mx, my - 0.5), _sample64(v, mx - 0.5, my)
        return x - dt / cell * vx, y - dt / cell * vy

    at = lambda n, m, ox, oy: (torch.arange(m, device="cuda", dtype=torch.float64)[None, :].expand(n, m) + ox,
                               torch.arange(n, device="cuda", dtype=torch.float64)[:, None].expand(n, m) + oy)
    for _ in range(steps):
        x, y = back(*at(h, w + 1, 0.0, 0.5))
        nu = _sample64(u, x, y - 0.5)
        x, y = back(*at(h + 1, w, 0.5, 0.0))
        nv = _sample64(v, x - 0.5, y)
        nu[:, 0] = nu[:, w] = 0.0
        nv[0] = nv[h] = 0.0
        nv[1:h] += wl.gravity_y * dt
        u, v, p = _poisson64(nu, nv, 100.0, cell, dt)
    return u, v, p


def _viscosity64(s):
    """M (x - x0) + dt K x = 0 on the interior faces, by CG with its diagonal, to 1e-11."""
    w, h, cell, dt = s["w"], s["h"], s["cell"], s["dt"]
    rho, mu = s["material"].view(h, w, 2).unbind(2)
    u0, v0 = s["u0"].view(h, w + 1), s["v0"].view(h + 1, w)
    mass_u, mass_v = torch.zeros_like(u0), torch.zeros_like(v0)
    mass_u[:, 1:w] = 0.5 * cell * cell * (rho[:, 1:] + rho[:, :-1])
    mass_v[1:h] = 0.5 * cell * cell * (rho[1:] + rho[:-1])
    corner = 0.25 * (mu[1:, 1:] + mu[1:, :-1] + mu[:-1, 1:] + mu[:-1, :-1])

    def apply(u, v):
        xx = 2.0 * mu * (u[:, 1:] - u[:, :-1])
        yy = 2.0 * mu * (v[1:] - v[:-1])
        shear = torch.zeros(h + 1, w + 1, dtype=torch.float64, device=u.device)
        shear[1:h, 1:w] = corner * ((u[1:, 1:w] - u[:-1, 1:w]) + (v[1:h, 1:] - v[1:h, :-1]))
        ku, kv = torch.zeros_like(u), torch.zeros_like(v)
        ku[:, 1:w] = (xx[:, :-1] - xx[:, 1:]) + (shear[:-1, 1:w] - shear[1:, 1:w])
        kv[1:h] = (yy[:-1] - yy[1:]) + (shear[1:h, :-1] - shear[1:h, 1:])
        return mass_u * u + dt * ku, mass_v * v + dt * kv

    pad = torch.zeros(h + 1, w + 1, dtype=torch.float64, device=mu.device)
    pad[1:h, 1:w] = corner
    du, dv = torch.ones_like(u0), torch.ones_like(v0)
    du[:, 1:w] = mass_u[:, 1:w] + dt * (2.0 * (mu[:, 1:] + mu[:, :-1]) + pad[:-1, 1:w] + pad[1:, 1:w])
    dv[1:h] = mass_v[1:h] + dt * (2.0 * (mu[1:] + mu[:-1]) + pad[1:h, :-1] + pad[1:h, 1:])
    inside_u, inside_v = (mass_u > 0).double(), (mass_v > 0).double()
    x = [u0 * inside_u, v0 * inside_v]
    a = apply(*x)
    r = [mass_u * u0 - a[0], mass_v * v0 - a[1]]
    z = [r[0] / du, r[1] / dv]
    d = [z[0].clone(), z[1].clone()]
    rz = (r[0] * z[0]).sum() + (r[1] * z[1]).sum()
    start = float(rz)
    for k in range(20000):
        if k % 100 == 0 and float(rz) <= 1e-22 * start:
            break
        q = apply(*d)
        alpha = rz / ((d[0] * q[0]).sum() + (d[1] * q[1]).sum())
        for i in (0, 1):
            x[i].add_(alpha * d[i])
            r[i].sub_(alpha * q[i])
        z = [r[0] / du, r[1] / dv]
        rz, last = (r[0] * z[0]).sum() + (r[1] * z[1]).sum(), rz
        for i in (0, 1):
            d[i].mul_(rz / last).add_(z[i])
    return x[0].reshape(-1), x[1].reshape(-1)


def _cuda(wl):
    w, h = wl.width, wl.height
    density = sum(m.reshape(-1, h, w).sum(0) for m in (wl.liquid_mass, wl.gas_mass)) / wl.cell_size ** 2
    solid = wl.meta.get("solid")
    return (torch.from_numpy(wl.u.reshape(h, w + 1)).cuda(), torch.from_numpy(wl.v.reshape(h + 1, w)).cuda(),
            torch.from_numpy(density).cuda(),
            None if solid is None else torch.from_numpy(solid.reshape(h, w) != 0).cuda())


def exact(case, seed):
    kind = case["kind"]
    if kind == "viscosity":
        u, v = _viscosity64(prepare(case, seed))
        return {"u": u, "v": v}
    if kind == "smoke":
        u, v, p = _smoke64(_workload(case, seed), case["steps"])
        return {"u": u.reshape(-1), "v": v.reshape(-1), "p": p.reshape(-1)}
    if kind == "project":
        wl = _workload(case, seed)
        u, v, density, solid = _cuda(wl)
        if case["scene"] == "vortex":
            u, v, p = _poisson64(u, v, 100.0, wl.cell_size, wl.dt)
        else:
            u, v, p = _project64(u, v, density, solid, wl.cell_size, wl.dt)
        result = {"u": u.reshape(-1), "v": v.reshape(-1)}
        return result if solid is not None else dict(result, p=p.reshape(-1))
    if kind == "batch":
        if case["count"] > 12:
            return None   # one small solve after another: minutes of launches
        parts = [_project64(*_cuda(wl), wl.cell_size, 1.0 / 240.0)
                 for wl in _instances(case, seed)]
        return {"u": torch.cat([a[0].reshape(-1) for a in parts]), "v": torch.cat([a[1].reshape(-1) for a in parts])}
    # advect: FP64 already, bit for bit the reference's expressions; step: the PLIC interface reconstruction and
    # the capillary fits of whole two-phase steps take minutes as tensor operations
    return None
