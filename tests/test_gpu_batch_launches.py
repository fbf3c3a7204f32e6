"""Batched projections over shapes at the edges of the shared launches: one tile, one row or column, one level, levels
that only the LDS tail takes, more tiles than are batched (solved on their own), with masks, both preconditioners,
several sweep counts, absolute and relative tolerances and spent budgets.  Every grid's result is fs_project's on the
same state bit for bit (the same kernels' arithmetic, the reductions per grid in the same order)."""
import time

import numpy as np
import pytest

from fluidsim_amd import FS_PRECOND_DIAGONAL, FS_PRECOND_MULTIGRID, FS_SMOOTHER_RED_BLACK, FluidGridHIP, batch_project
from fluidsim_amd import workloads as WL

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (8, 8), (2, 1), (1, 130), (64, 16), (65, 17), (9, 9), (200, 20), (129, 65), (61, 47), (300, 111), (70, 58),
          (1000, 1100), (257, 90)]


def grids():
    out = []
    for k, (W, H) in enumerate(SHAPES):
        wl = WL.sloped_pool(W, H, 4.0)
        g = FluidGridHIP(W, H, 4.0)
        WL.load_into(g, wl)
        if k % 3 == 0 and W > 8 and H > 8:
            solid = np.zeros((H, W), np.uint8)
            solid[H // 3:H // 3 + 3, W // 4:W // 4 + 5] = 1
            g.setSolidMask(solid)
        if k % 4 == 1:
            g.setPressurePreconditioner(FS_PRECOND_DIAGONAL)
        if k % 2:
            g.setPressureSmoother(FS_SMOOTHER_RED_BLACK, 1 + k % 4, 1 + k % 3)
        if k % 5 == 2:
            g.setRelativeTolerance(True)
        g.snapshotSave()
        out.append(g)
    return out


def state(g):
    s = g.download()
    return s.u, s.v, s.pressure


@pytest.mark.parametrize("budget", [3, 400])
def test_batched_projections_are_the_single_ones(budget):
    many, dt = grids(), 1.0 / 120.0
    expected = []
    for rounds in (1, 2):   # the second from the first one's pressure, its hierarchy still valid
        for g in many:
            if rounds == 1:
                g.snapshotRestore()
            else:
                g.addVortex((4.0, 4.0), 20.0, 0.1)
            r = g.project(dt, budget, 1e-5)
            expected.append((r, state(g)))
    at = 0
    for rounds in (1, 2):
        for g in many:
            if rounds == 1:
                g.snapshotRestore()
            else:
                g.addVortex((4.0, 4.0), 20.0, 0.1)
        results = batch_project(many, dt, budget, 1e-5)
        for g, r in zip(many, results):
            ref, fields = expected[at]
            at += 1
            key = (rounds, g.width, g.height)
            assert (r.iterations, r.converged, r.restarts) == (ref.iterations, ref.converged, ref.restarts), key
            assert r.max_divergence == ref.max_divergence and r.final_residual == ref.final_residual, key
            for a, b in zip(state(g), fields):
                assert np.array_equal(a, b), key
    for g in many:
        g.destroy()


@pytest.mark.parametrize("precond", [FS_PRECOND_DIAGONAL, FS_PRECOND_MULTIGRID])
def test_small_checks_across_refreshed_residuals(precond):
    """Grids of one to four tiles, whose check and decision share a launch of up to sixteen wavefronts, through solves that
    refresh the residual every 32 iterations many times over: the batch's separate launches give the same bits,
    time after time."""
    many, dt = [], 1.0 / 120.0
    for W, H in [(61, 47), (64, 64), (128, 32), (130, 10), (256, 16), (33, 16), (64, 17)]:
        wl = WL.sloped_pool(W, H, 4.0)
        g = FluidGridHIP(W, H, 4.0)
        WL.load_into(g, wl)
        g.setPressurePreconditioner(precond)
        g.snapshotSave()
        many.append(g)
    expected = None
    for _ in range(4):
        got = []
        for g in many:
            g.snapshotRestore()
            r = g.project(dt, 3000, 1e-9)
            got.append((r.iterations, r.restarts, r.final_residual, r.max_divergence) + state(g))
        for g in many:
            g.snapshotRestore()
        for g, r in zip(many, batch_project(many, dt, 3000, 1e-9)):
            got.append((r.iterations, r.restarts, r.final_residual, r.max_divergence) + state(g))
        n = len(many)
        if precond == FS_PRECOND_DIAGONAL:
            assert max(x[0] for x in got[:n]) > 100
        for a, b in zip(got[:n], got[n:]):
            assert all(np.array_equal(x, y) for x, y in zip(a, b))
        expected = expected or got
        for a, b in zip(got, expected):
            assert all(np.array_equal(x, y) for x, y in zip(a, b))
    for g in many:
        g.destroy()


def test_grids_of_one_level_share_launches():
    """Sixteen 8 x 8 grids in a batch take little longer than two (one after another they would take eight times as long)."""
    def fastest(n):
        many = []
        for _ in range(n):
            wl = WL.sloped_pool(8, 8, 4.0)
            g = FluidGridHIP(8, 8, 4.0)
            WL.load_into(g, wl)
            many.append(g)
        times = []
        for _ in range(8):
            t = time.perf_counter()
            batch_project(many, 1.0 / 120.0, 20, 1e-5)
            times.append(time.perf_counter() - t)
        for g in many:
            g.destroy()
        return min(times)
    assert fastest(16) < 4.0 * fastest(2)
