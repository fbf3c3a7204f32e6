"""Batched timesteps on the GPU (fs_batch_step) and the serving loop's batched route.

fs_batch_step is fs_step on many grids at once, each with its own dt, budget and tolerance; its viscosity
solves run in one persistent launch and its projections in launches shared by all grids.  Checked here:
  - each grid's step agrees with fs_step on a copy: the fractions bit for bit after the first step
    (transport runs first, from the same state), velocities to the batched solves' rounding, iteration
    counts within a few, and every projection converges;
  - a grid's result is the same alone and in any batch, bit for bit;
  - per-grid dt <= 0 leaves that grid untouched (physical_steps 0), and a grid that fails (a capillary
    substep count beyond the int range) is reported in its own status while the others step normally;
  - a server with batch_cells steps its small requests through fs_batch_step: each served result equals the
    request stepped by fs_batch_step alone (small) or by fs_step (larger) on a plain grid, bit for bit.
"""
import numpy as np
import pytest

from fluidsim_amd import FS_TRANSPORT_REFERENCE, FluidGridHIP, FluidGridState, FluidMixture, MixtureComponent
from fluidsim_amd import batch_step
from fluidsim_amd import workloads as WL
from fluidsim_amd.serving import Request, Server

pytestmark = pytest.mark.gpu

FS_OK, FS_E_RUNTIME = 0, 5

# (W, H, kinematic viscosity, surface tension, dt)
CASES = [(40, 30, 0.0, 0.0, 0.002), (64, 64, 0.01, 0.0, 0.0015), (100, 70, 0.0, 0.03, 0.001),
         (128, 96, 0.1, 0.02, 0.001), (33, 129, 0.002, 0.0, 0.002), (200, 150, 0.05, 0.05, 0.0005)]


def make(W, H, nu, sigma, seed):
    rng = WL.SplitMix64(seed)
    h = 1.0 / max(W, H)
    f = WL.pool_with_drop(W, H, h, 0.35 + 0.5 * rng.uniform(1)[0], 0.1, rng)
    u = np.zeros((W + 1) * H)
    v = np.zeros(W * (H + 1))
    for _ in range(5):
        WL.add_gaussian(u, v, W, H, h, rng.uniform(1, 0, W * h)[0], rng.uniform(1, 0, H * h)[0],
                        rng.uniform(1, 0.03, 0.08)[0], 0.3 * rng.normal(1)[0])
    WL.zero_walls(u, v, W, H)
    lm, gm = WL.two_phase_masses(f, h)
    g = FluidGridHIP(W, H, h)
    g.configureMaterials([], FluidMixture([MixtureComponent("water", 100.0, nu * 100.0)]),
                         FluidMixture([MixtureComponent("air", 0.1, nu * 0.1)]))
    g.setGravityY(9.81)
    g.setSurfaceTension(sigma)
    g.setTransport(FS_TRANSPORT_REFERENCE)
    g.upload(FluidGridState(f, u, v, np.zeros(0), [lm], [gm]))
    return g


def grids_of(cases):
    return [make(W, H, nu, sigma, k) for k, (W, H, nu, sigma, _) in enumerate(cases)]


def test_batch_step_agrees_with_single_steps():
    batch, single = grids_of(CASES), grids_of(CASES)
    dts = [c[4] for c in CASES]
    scales = []
    for g in batch:
        s = g.download()
        scales.append(max(np.abs(s.u).max(), np.abs(s.v).max()))
    for step in range(3):
        res, statuses = batch_step(batch, dts, 2000, 1e-6)
        assert statuses == [FS_OK] * len(CASES)
        for k, (g, s) in enumerate(zip(batch, single)):
            r = res[k]
            rs = s.step(dts[k], 2000, 1e-6)
            name = f"{CASES[k][:2]} step {step}"
            assert r.converged and rs.converged, (name, r, rs)
            assert r.physical_steps == rs.physical_steps >= 1, name
            assert abs(r.iterations - rs.iterations) <= 3 * r.physical_steps, (name, r.iterations, rs.iterations)
            assert abs(r.viscosity_iterations - rs.viscosity_iterations) <= 4 * r.physical_steps, name
            assert (r.viscosity_iterations > 0) == (CASES[k][2] > 0), name
            a, b = g.download(), s.download()
            if step == 0:
                assert np.array_equal(a.liquid_fraction, b.liquid_fraction), name
            tol = 1e-3 * scales[k] * (step + 1)
            assert np.abs(a.u - b.u).max() <= tol and np.abs(a.v - b.v).max() <= tol, name
    for g in batch + single:
        g.destroy()


def test_alone_equals_in_any_batch():
    grids = grids_of(CASES)
    dts = [c[4] for c in CASES]
    k = 3
    alone = make(*CASES[k][:4], k)
    for _ in range(2):
        res, _ = batch_step(grids, dts, 2000, 1e-6)
        ra, _ = batch_step([alone], dts[k], 2000, 1e-6)
        r = res[k]
        assert (r.iterations, r.viscosity_iterations, r.max_divergence) == \
               (ra[0].iterations, ra[0].viscosity_iterations, ra[0].max_divergence)
    s, sa = grids[k].download(), alone.download()
    for key in ("liquid_fraction", "u", "v", "pressure"):
        assert np.array_equal(getattr(s, key), getattr(sa, key)), key
    for g in grids + [alone]:
        g.destroy()


def test_zero_dt_and_a_failing_grid_stay_per_grid():
    cases = CASES[:4]
    grids = grids_of(cases)
    refs = grids_of(cases)
    before = grids[0].download()
    # grid 0: dt = 0 (untouched); grid 2: surface tension asks for more capillary substeps than an int holds
    dts = [0.0, cases[1][4], 1e30, cases[3][4]]
    res, statuses = batch_step(grids, dts, 2000, 1e-6, raise_on_error=False)
    assert statuses == [FS_OK, FS_OK, FS_E_RUNTIME, FS_OK]
    assert res[0].physical_steps == 0 and not res[0].converged
    after = grids[0].download()
    assert np.array_equal(after.u, before.u) and np.array_equal(after.liquid_fraction, before.liquid_fraction)
    assert res[2].physical_steps == 0
    with pytest.raises(RuntimeError, match="capillary|substeps"):
        batch_step(grids[2:3], [1e30], 2000, 1e-6)
    # the healthy grids equal the same grids stepped without the others
    ok = [1, 3]
    rr, _ = batch_step([refs[i] for i in ok], [dts[i] for i in ok], 2000, 1e-6)
    for j, i in enumerate(ok):
        assert res[i].converged and (res[i].iterations, res[i].max_divergence) == (rr[j].iterations, rr[j].max_divergence)
        assert np.array_equal(grids[i].download().u, refs[i].download().u)
    for g in grids + refs:
        g.destroy()


def request(W, H, seed, steps=4, nu=0.0, sigma=0.0):
    rng = WL.SplitMix64(seed)
    h = 1.0 / max(W, H)
    f = WL.pool_with_drop(W, H, h, 0.5, 0.1, rng)
    u = np.zeros((W + 1) * H)
    v = np.zeros(W * (H + 1))
    for _ in range(4):
        WL.add_gaussian(u, v, W, H, h, rng.uniform(1, 0, W * h)[0], rng.uniform(1, 0, H * h)[0], 0.05,
                        0.2 * rng.normal(1)[0])
    WL.zero_walls(u, v, W, H)
    lm, gm = WL.two_phase_masses(f, h)
    return Request(width=W, height=H, cell_size=h, steps=steps, dt=0.0015, max_iterations=-1,
                   divergence_tolerance=1e-6, relative_tolerance=True, gravity_y=9.81, surface_tension=sigma,
                   liquid_viscosity=[nu * 100.0], gas_viscosity=[nu * 0.1], liquid_fraction=f, u=u, v=v,
                   liquid_mass=lm, gas_mass=gm)


def plain(r: Request, batched: bool):
    """The request stepped on a plain grid: by fs_batch_step alone, or by fs_step."""
    g = FluidGridHIP(r.width, r.height, r.cell_size)
    g.configureMaterials([], FluidMixture([MixtureComponent("water", 100.0, r.liquid_viscosity[0])]),
                         FluidMixture([MixtureComponent("air", 0.1, r.gas_viscosity[0])]))
    g.setGravityY(r.gravity_y)
    g.setSurfaceTension(r.surface_tension)
    g.setRelativeTolerance(True)
    g.upload(FluidGridState(r.liquid_fraction, r.u, r.v, np.zeros(0), [r.liquid_mass], [r.gas_mass]))
    pressure = viscosity = 0
    for _ in range(r.steps):
        if batched:
            (res,), _ = batch_step([g], r.dt, r.max_iterations, r.divergence_tolerance)
        else:
            res = g.step(r.dt, r.max_iterations, r.divergence_tolerance)
        assert res.accepted()
        pressure += res.iterations
        viscosity += res.viscosity_iterations
    s = g.download()
    g.destroy()
    return s, pressure, viscosity


def test_server_batches_small_requests():
    limit = 100 * 100
    reqs = [request(96, 64, 1, nu=0.01), request(300, 200, 2, nu=0.05, sigma=0.03), request(64, 64, 3, sigma=0.02),
            request(100, 100, 4, nu=0.1), request(180, 120, 5), request(40, 128, 6, nu=0.002, sigma=0.01),
            request(256, 128, 7, nu=0.02)]
    assert 0 < sum(r.width * r.height <= limit for r in reqs) < len(reqs)
    with Server(lanes=2, batch_cells=limit) as srv:
        ids = [srv.submit(r) for r in reqs]
        srv.drain()
        reps = [srv.wait(i) for i in ids]
        outs = [srv.result(i, r.width, r.height) for i, r in zip(ids, reqs)]
        st = srv.stats()
    assert st["completed"] == len(reqs) and st["failed"] == 0
    # small and larger requests are each spread over both lanes
    small = [rep.lane for rep, r in zip(reps, reqs) if r.width * r.height <= limit]
    large = [rep.lane for rep, r in zip(reps, reqs) if r.width * r.height > limit]
    assert set(small) == {0, 1} and set(large) == {0, 1}
    for rep, out, r in zip(reps, outs, reqs):
        name = f"{r.width}x{r.height}"
        assert rep.done and rep.steps_done == r.steps, (name, rep.error)
        s, pressure, viscosity = plain(r, r.width * r.height <= limit)
        assert (rep.pressure_iterations, rep.viscosity_iterations) == (pressure, viscosity), name
        for key, got in (("fraction", s.liquid_fraction), ("u", s.u), ("v", s.v), ("pressure", s.pressure)):
            assert np.array_equal(out[key], got), f"{name}: {key}"
