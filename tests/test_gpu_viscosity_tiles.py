"""The viscosity solve's register kernels (descent, ascent, operator tiles, one-workgroup tail) at the sizes where they
can go wrong: one level, tiles filled exactly and by one slot more, a tail of one to four levels and at its slot
limit, the tile heights chosen for small and large levels with each smoother.

Reference: the FP64 oracle with the same smoother.  The recomputed residual after one, two and four iterations shows a
wrong sweep, halo or transfer at once: without the last tap of the last coarse column the oracle's own changes by 2e-4
to 3, and here FP32 moves it by eight bits of rounding (measured at most 2e-5 of the residual, and 2e-7 of the velocity
scale where little is left).  The other smoothers, which no entry point stops early, are held by their solves: on grids
where rounding costs no iteration the counts are the oracle's and the velocities within 2e-5 of the scale (measured at
most 7e-6; the same planted mistake moves the 62 x 62 and 123 x 33 ones by 4e-5 to 1.4e-4); thin and large ones, whose
FP32 recurrence needs up to half as many iterations again, within 1e-4 (measured at most 2e-5, and the mistake triples
the counts of thin ones).

Also against fs_batch_apply_viscosity, which runs every level as plain loops over the slots in memory.  Both stop at a
relative residual of 1e-4 looked at every four iterations, so the counts agree to one look and the velocities to
that tolerance times the ten that the batched and single solves are held to elsewhere."""
import ctypes as C

import numpy as np
import pytest

from fluidsim_amd import (FS_TRANSPORT_NONE, FluidGridHIP, FluidGridState, FluidMixture, MixtureComponent, _abi,
                          batch_apply_viscosity, default_context)
from fluidsim_amd import workloads as WL

pytestmark = pytest.mark.gpu


def viscous(W, H, sweeps):
    rng = WL.SplitMix64(31)
    h, nu = 1.0 / max(W, H), 0.1
    f = WL.pool_with_drop(W, H, h, 0.5, 0.1, rng)
    u, v = rng.normal((W + 1) * H), rng.normal(W * (H + 1))
    WL.zero_walls(u, v, W, H)
    lm, gm = WL.two_phase_masses(f, h)
    g = FluidGridHIP(W, H, h)
    g.configureMaterials([], FluidMixture([MixtureComponent("water", 100.0, nu * 100.0)]),
                         FluidMixture([MixtureComponent("air", 0.1, nu * 0.1)]))
    g.setTransport(FS_TRANSPORT_NONE)
    g.setViscositySmoother(sweeps)
    g.upload(FluidGridState(f, u, v, np.zeros(0), [lm], [gm]))
    return g


SMALL = [(1, 1), (8, 8), (64, 1), (1, 64), (9, 8), (55, 7), (56, 8), (57, 15), (59, 11), (60, 12), (62, 62), (63, 62),
         (111, 24), (123, 33)]
THIN_OR_LARGE = [(1022, 1), (2, 700), (1024, 512)]


@pytest.mark.parametrize("W,H", SMALL + THIN_OR_LARGE)
def test_residuals_of_the_first_iterations_are_the_oracles(oracle, W, H):
    g = viscous(W, H, 0)
    s = g.download()
    g.destroy()
    h, dt = 1.0 / max(W, H), 0.002
    material = oracle.viscosity_material(h, [100.0], [10.0], s.liquid_mass[0], [0.1], [0.01], s.gas_mass[0], W * H)
    m = np.ascontiguousarray(material, dtype=np.float64).ravel()
    for budget in (1, 2, 4):
        u, v = s.u.copy(), s.v.copy()
        n, rel = C.c_int(), C.c_double()
        dp = C.POINTER(C.c_double)
        _abi.lib().fs_viscosity_solve(default_context().handle, W, H, h, m.ctypes.data_as(dp), u.ctypes.data_as(dp),
                                      v.ctypes.data_as(dp), dt, 1e-30, budget, C.byref(n), C.byref(rel))
        _, on, orel, _, _ = oracle.viscosity_solve(W, H, h, material, s.u, s.v, dt, 1e-30, budget)
        assert n.value == on, budget
        assert abs(rel.value - orel) <= 6e-5 * orel + 6e-7, (budget, rel.value, orel)


def solved(oracle, W, H, sweeps, dt):
    g = viscous(W, H, sweeps)
    s = g.download()
    o = oracle.OracleGrid(W, H, 1.0 / max(W, H))
    o.configure([100.0], [0.1])
    o.configure_viscosity([10.0], [0.01])
    o.set_viscosity_smoother(sweeps)
    o.upload(s.liquid_fraction, s.u, s.v, None, s.liquid_mass[0], s.gas_mass[0])
    status, on = o.apply_viscosity(dt)
    assert status == oracle.VISC_OK
    n = g.applyViscosity(dt)
    a, b = g.download(), o.download()
    g.destroy()
    scale = max(np.abs(s.u).max(), np.abs(s.v).max(), 1e-12)
    return n, on, max(np.abs(a.u - b["u"]).max(), np.abs(a.v - b["v"]).max()) / scale


@pytest.mark.parametrize("W,H", SMALL)
@pytest.mark.parametrize("sweeps", [2, 4, 6])
def test_smoothers_match_the_oracle(oracle, W, H, sweeps):
    n, on, error = solved(oracle, W, H, sweeps, 0.02)
    assert n == on and error <= 2e-5, (n, on, error)


@pytest.mark.parametrize("W,H", THIN_OR_LARGE)
@pytest.mark.parametrize("sweeps", [0, 4, 6])
def test_smoothers_match_the_oracle_on_thin_and_large_grids(oracle, W, H, sweeps):
    n, on, error = solved(oracle, W, H, sweeps, 0.002)
    assert n <= 1.5 * on + 4 and error <= 1e-4, (n, on, error)


@pytest.mark.parametrize("W,H", SMALL + THIN_OR_LARGE)
@pytest.mark.parametrize("sweeps", [0, 4, 6])
def test_single_solves_match_the_batched_loops(W, H, sweeps):
    check(W, H, sweeps)


def test_large_levels_with_six_sweeps():
    check(1030, 1020, 6)


def check(W, H, sweeps):
    dt = 0.002
    a, b = viscous(W, H, sweeps), viscous(W, H, sweeps)
    n = a.applyViscosity(dt)
    m = batch_apply_viscosity([b], dt)[0]
    assert abs(n - m) <= 4, (n, m)
    sa, sb = a.download(), b.download()
    scale = max(np.abs(sb.u).max(), np.abs(sb.v).max(), 1e-12)
    assert np.abs(sa.u - sb.u).max() <= 1e-3 * scale and np.abs(sa.v - sb.v).max() <= 1e-3 * scale
    a.destroy()
    b.destroy()
