"""Every launch choice of the level smoothers on grids whose edges fall inside, on and just past the tiles' interiors,
with every sweep count and storage type, with and without solid cells: the same V-cycle bit for bit, and for FP32
levels the oracle's within 1e-5 (FP32 smoothing against FP64: the bar of the smoother tests).
"""
import numpy as np
import pytest

from fluidsim_amd import (FS_MG_BF16, FS_MG_BF16_VECTORS, FS_MG_FP16, FS_MG_FP32, FS_SMOOTHER_CHEBYSHEV,
                          FS_SMOOTHER_RED_BLACK, FluidGridHIP)
from fluidsim_amd import workloads as WL

pytestmark = pytest.mark.gpu


@pytest.fixture
def O(oracle):
    yield oracle
    oracle.set_smoother(oracle.SMOOTH_RBGS, 4)


def tank(W, H, solids):
    rng = WL.SplitMix64(W + H)
    wl = WL.sloped_pool(W, H, 4.0)
    solid = None
    if solids:
        # isolated 1 x 2 blocks: connected fluid, cells without conductance on every level's edge
        solid = np.zeros((H, W), np.uint8)
        for x, y in zip((rng.uniform(12) * (W // 4)).astype(int) * 4, (rng.uniform(12) * (H // 4)).astype(int) * 4):
            solid[y:y + 1, x:x + 2] = 1
        solid = solid.ravel()
        wl.fraction[solid != 0] = 0.0
        wl.liquid_mass, wl.gas_mass = WL.two_phase_masses(wl.fraction, wl.cell_size)
    return wl, solid


def grid(wl, solid):
    g = FluidGridHIP(wl.width, wl.height, wl.cell_size)
    WL.load_into(g, wl)
    if solid is not None:
        g.setSolidMask(solid)
    return g


SHAPES = [(129, 65), (67, 150), (112, 96), (225, 97), (90, 301)]
CHOICES = [(FS_SMOOTHER_RED_BLACK, 1), (FS_SMOOTHER_RED_BLACK, 3), (FS_SMOOTHER_RED_BLACK, 4),
           (FS_SMOOTHER_CHEBYSHEV, 1), (FS_SMOOTHER_CHEBYSHEV, 2), (FS_SMOOTHER_CHEBYSHEV, 7), (FS_SMOOTHER_CHEBYSHEV, 8)]


@pytest.mark.parametrize("solids", [False, True])
@pytest.mark.parametrize("W,H", SHAPES)
def test_every_choice_is_the_same_vcycle(O, W, H, solids):
    wl, solid = tank(W, H, solids)
    g = grid(wl, solid)
    o = O.OracleGrid(W, H, wl.cell_size)
    o.configure(wl.liquid_density, wl.gas_density)
    if solid is not None:
        o.set_solid(solid)
    o.upload(wl.fraction, wl.u, wl.v, None, wl.liquid_mass, wl.gas_mass)
    i = np.arange(W * H)
    a = np.sin(i * 0.31) + np.cos(i * 0.073)
    if solid is not None:
        a *= solid == 0
    a -= a.mean()
    for kind, sweeps in CHOICES:
        g.setPressureSmoother(kind, sweeps, 4)
        O.set_smoother(kind, sweeps, 4)
        o.project(wl.dt, 0, 1.0)
        g.project(wl.dt, 0, 1.0)
        expected = o.multigrid().apply(a, 0.0)
        levels = [l for l in range(g.multigridLevels()) if g.multigridTiles(l)[0] >= 0]
        cheb = [kind == FS_SMOOTHER_CHEBYSHEV and np.prod(g.multigridShape(l)) > 4096 for l in levels]
        reference = None
        for v in range(11):
            for l, c in zip(levels, cheb):
                g.setMultigridTiles(l, v, v % 8 if c else v, v % 4)
            out = g.multigridApply(a)
            if reference is None:
                reference = out
                assert np.linalg.norm(out - expected) < 1e-5 * np.linalg.norm(expected), (kind, sweeps)
            assert np.array_equal(out, reference), (kind, sweeps, v)
    g.destroy()


@pytest.mark.parametrize("mode", [FS_MG_FP16, FS_MG_BF16, FS_MG_BF16_VECTORS])
@pytest.mark.parametrize("W,H", SHAPES)
def test_every_choice_is_the_same_16_bit_vcycle(W, H, mode):
    wl, solid = tank(W, H, True)
    g = grid(wl, solid)
    i = np.arange(W * H)
    a = (np.sin(i * 0.31) + np.cos(i * 0.073)) * (solid == 0)
    a -= a.mean()
    full = g.multigridApply(a)
    g.setMultigridPrecision(mode)
    levels = [l for l in range(g.multigridLevels()) if g.multigridTiles(l)[0] >= 0]
    reference = None
    for v in range(11):
        for l in levels:
            g.setMultigridTiles(l, v, v, v % 4)
        out = g.multigridApply(a)
        reference = out if reference is None else reference
        assert np.array_equal(out, reference), v
    # rounding the conductances moves the V-cycle by their relative error, 2^-11 or 2^-8, vectors by 2^-8 a store
    assert np.linalg.norm(reference - full) < (2e-3 if mode == FS_MG_FP16 else 3e-2) * np.linalg.norm(full)
    g.destroy()


@pytest.mark.parametrize("coarse", [1, 4])
@pytest.mark.parametrize("W,H", [(64, 64), (63, 65), (65, 33), (70, 58), (66, 62), (128, 32), (129, 31), (200, 20), (2, 700),
                                 (9, 9), (12, 7), (31, 130), (33, 17)])
def test_coarse_levels_match_the_oracle(O, W, H, coarse):
    """Grids whose levels all run in the single-workgroup tail: two, four and eight rows per thread, one to four levels
    above the coarsest, and shapes its register layout does not take (more than 128 columns)."""
    wl, _ = tank(W, H, False)
    g = grid(wl, None)
    g.setPressureSmoother(FS_SMOOTHER_RED_BLACK, 4, coarse)
    O.set_smoother(FS_SMOOTHER_RED_BLACK, 4, coarse)
    o = O.OracleGrid(W, H, wl.cell_size)
    o.configure(wl.liquid_density, wl.gas_density)
    o.upload(wl.fraction, wl.u, wl.v, None, wl.liquid_mass, wl.gas_mass)
    o.project(wl.dt, 0, 1.0)
    g.project(wl.dt, 0, 1.0)
    i = np.arange(W * H)
    a = np.sin(i * 0.31) + np.cos(i * 0.073)
    a -= a.mean()
    expected, out = o.multigrid().apply(a, 0.0), g.multigridApply(a)
    assert np.linalg.norm(out - expected) < 1e-5 * np.linalg.norm(expected)
    g.destroy()
