"""Semi-Lagrangian transport at the edges of its 256-element workgroups, on rows of one and two elements, of powers of two
and next to them (an element's row is found by a multiplication) and on a very tall grid, with velocities that leave the
grid: bit for bit the FP64 oracle's.  Narrow grids take no longer than square ones of as many cells."""
import time

import numpy as np
import pytest

from fluidsim_amd import Context, FluidGridHIP, FluidGridState, FluidMixture, MixtureComponent

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,cell", [(1, 1, 1.0), (63, 4, 0.1), (64, 5, 0.25), (65, 3, 4.0), (200, 1, 0.3), (1, 130, 1.0),
                                      (3, 1000, 0.2), (7, 700, 0.4), (255, 33, 0.1), (256, 3, 1.0), (257, 129, 0.2),
                                      (2, 262200, 0.5)])
def test_semi_lagrangian_at_tile_edges_is_bitwise(oracle, W, H, cell):
    rng = np.random.default_rng(W + H)
    f = np.clip(rng.uniform(-0.5, 1.5, W * H), 0.0, 1.0)
    u, v = rng.normal(size=(W + 1) * H) * 3.0 * cell, rng.normal(size=W * (H + 1)) * 3.0 * cell
    u[::7], v[::5] = 0.0, 0.0
    lm, gm = 100.0 * cell * cell * f, 0.1 * cell * cell * (1.0 - f)
    g = FluidGridHIP(W, H, cell)
    g.configureMaterials([], FluidMixture([MixtureComponent("l", 100.0)]), FluidMixture([MixtureComponent("g", 0.1)]))
    g.upload(FluidGridState(f, u, v, np.zeros(0), [lm], [gm]))
    o = oracle.OracleGrid(W, H, cell)
    o.configure([100.0], [0.1])
    o.upload(f, u, v, None, lm, gm)
    g.advectSemiLagrangian(1.3)
    o.advect_semi_lagrangian(1.3)
    a, b = g.download(), o.download()
    g.destroy()
    for name, got in (("fraction", a.liquid_fraction), ("u", a.u), ("v", a.v), ("liquid_mass", a.liquid_mass[0]),
                      ("gas_mass", a.gas_mass[0])):
        assert np.array_equal(got, b[name]), name


def test_narrow_grids_keep_the_lanes_busy():
    def fastest(W, H):
        ctx = Context(0)
        f = np.ones(W * H)
        g = FluidGridHIP(W, H, 1.0, context=ctx)
        g.configureMaterials([], FluidMixture([MixtureComponent("l", 100.0)]), FluidMixture([MixtureComponent("g", 0.1)]))
        g.upload(FluidGridState(f, np.zeros((W + 1) * H), np.zeros(W * (H + 1)), np.zeros(0), [100.0 * f], [0.0 * f]))
        times = []
        for _ in range(6):
            ctx.synchronize()
            t = time.perf_counter()
            for _ in range(20):
                g.advectSemiLagrangian(0.1)
            ctx.synchronize()
            times.append(time.perf_counter() - t)
        g.destroy()
        ctx.close()
        return min(times)
    assert fastest(2, 100000) < 2.5 * fastest(447, 447)
