"""The viscosity solve's register kernels (descent, ascent, operator tiles, one-workgroup tail) at the sizes where they
can go wrong: one level, tiles filled exactly and by one slot more, a tail of one to four levels and at its slot
limit, the tile heights chosen for small and large levels with each smoother.  Reference: fs_batch_apply_viscosity, which
runs every level as plain loops over the slots in memory.  Both stop at a relative residual of 1e-4 looked at every
four iterations, so the counts agree to one look (a wrong transfer or sweep costs CG more) and the velocities to
that tolerance times the ten that the batched and single solves are held to elsewhere."""
import numpy as np
import pytest

from fluidsim_amd import (FS_TRANSPORT_NONE, FluidGridHIP, FluidGridState, FluidMixture, MixtureComponent,
                          batch_apply_viscosity)
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


@pytest.mark.parametrize("W,H", [(1, 1), (8, 8), (64, 1), (1, 64), (9, 8), (55, 7), (56, 8), (57, 15), (59, 11), (60, 12),
                                 (62, 62), (63, 62), (111, 24), (123, 33), (1022, 1), (2, 700), (1024, 512)])
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
