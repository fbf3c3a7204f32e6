"""Semi-Lagrangian transport at the edges of its 64 x 4 workgroups and beyond the rows one launch covers (65535 x 4), with
velocities that leave the grid: bit for bit the FP64 oracle's."""
import numpy as np
import pytest

from fluidsim_amd import FluidGridHIP, FluidGridState, FluidMixture, MixtureComponent

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,cell", [(1, 1, 1.0), (63, 4, 0.1), (64, 5, 0.25), (65, 3, 4.0), (200, 1, 0.3), (1, 130, 1.0),
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
