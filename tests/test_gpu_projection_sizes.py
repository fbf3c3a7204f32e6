"""Projections at the edges of the PCG kernels' tiles: 64 x 16 cells per tile, one or four tiles per workgroup
(more than 1024 tiles in more than one row), pre-reduced partials (more than 1024 workgroups), grids of one row or
column.

One constant density, so the Neumann problem is diagonal in cosines and the exact velocity is known in 64 bits.
A solve that stops at max|b - A p| <= tol max|b| leaves, with L the unit-weight Laplacian (L = G^T G, G the face
differences) and w the face weight, a pressure error L^-1 r / w and a velocity error (dt / h) G L^-1 r of 2-norm at most
(dt / h) sqrt(n) tol max|b| / sqrt(lambda), lambda = 2 - 2 cos(pi / max(W, H)) the smallest nonzero eigenvalue of L.
"""
import numpy as np
import pytest
from scipy.fft import dctn, idctn

from fluidsim_amd import FS_SMOOTHER_CHEBYSHEV, FS_SMOOTHER_RED_BLACK, FluidGridHIP
from fluidsim_amd import workloads as WL

pytestmark = pytest.mark.gpu

TOL = 1e-7


def box(W, H, seed):
    rng = WL.SplitMix64(seed)
    h = 1.0 / max(W, H)
    u, v = rng.normal((W + 1) * H), rng.normal(W * (H + 1))
    WL.zero_walls(u, v, W, H)
    fraction = np.ones(W * H)
    liquid, gas = WL.two_phase_masses(fraction, h)
    return WL.Workload("box", W, H, h, [100.0], [0.1], 9.81, 1.0 / 120.0, fraction, u, v, liquid, gas)


def exact(wl):
    W, H, h, dt = wl.width, wl.height, wl.cell_size, wl.dt
    u, v = wl.u.reshape(H, W + 1).copy(), wl.v.reshape(H + 1, W).copy()
    b = -((u[:, 1:] - u[:, :-1]) + (v[1:] - v[:-1])) / h * (h * h / dt)
    symbol = ((2.0 - 2.0 * np.cos(np.pi * np.arange(W) / W))[None, :] +
              (2.0 - 2.0 * np.cos(np.pi * np.arange(H) / H))[:, None]) / 100.0
    symbol[0, 0] = 1.0
    spectrum = dctn(b, type=2) / symbol
    spectrum[0, 0] = 0.0
    p = idctn(spectrum, type=2)
    u[:, 1:W] -= (p[:, 1:] - p[:, :-1]) / h * dt / 100.0
    v[1:H] -= (p[1:] - p[:-1]) / h * dt / 100.0
    lam = 2.0 - 2.0 * np.cos(np.pi / max(W, H))
    bound = dt / h * np.sqrt(W * H) * TOL * np.abs(b).max() / np.sqrt(lam)
    return u.ravel(), v.ravel(), bound


@pytest.mark.parametrize("smoother", [(FS_SMOOTHER_RED_BLACK, 4, 4), (FS_SMOOTHER_CHEBYSHEV, 3, 2)])
@pytest.mark.parametrize("W,H", [(2, 1), (1, 130), (64, 16), (65, 17), (63, 145), (300, 111), (1025, 1030),
                                 (2112, 2050), (66000, 3), (35000, 20), (22000, 40)])
def test_projection_matches_the_exact_one(W, H, smoother):
    wl = box(W, H, 7 * W + H)
    eu, ev, bound = exact(wl)
    g = FluidGridHIP(W, H, wl.cell_size)
    WL.load_into(g, wl)
    g.setPressureSmoother(*smoother)
    g.setRelativeTolerance(True)
    res = g.project(wl.dt, 200, TOL)
    s = g.download()
    assert res.converged
    error = np.hypot(np.linalg.norm(s.u - eu), np.linalg.norm(s.v - ev))
    assert error <= bound + 1e-12 * np.hypot(np.linalg.norm(eu), np.linalg.norm(ev))
    g.destroy()


@pytest.mark.parametrize("budget", [0, 1, 3])
def test_a_spent_budget_stops_the_solve(budget):
    wl = box(130, 70, 3)
    g = FluidGridHIP(wl.width, wl.height, wl.cell_size)
    WL.load_into(g, wl)
    g.setRelativeTolerance(True)
    res = g.project(wl.dt, budget, 1e-14)
    assert not res.converged and res.iterations == budget
    g.destroy()


def test_a_single_tile_reduces_no_partials_apart():
    """The update of a grid of one 64 x 16 tile is one launch, as on a grid of two (a second one, reducing the single
    partial into itself, would double it)."""
    def fastest(H):
        wl = box(64, H, 5)
        g = FluidGridHIP(64, H, wl.cell_size)
        WL.load_into(g, wl)
        g.project(wl.dt, 3, TOL)
        ms = min(g.timeKernel(2, 500) for _ in range(8))
        g.destroy()
        return ms
    one, two = fastest(16), fastest(17)
    assert one < 1.4 * two, (one, two)


def test_flat_grids_visit_no_empty_tiles():
    """r.z of a grid of one row of 1563 tiles is a launch over them and one that reduces their partials: less than twice
    what a square grid of about as many cells takes for the first alone."""
    def fastest(W, H):
        wl = box(W, H, 5)
        g = FluidGridHIP(W, H, wl.cell_size)
        WL.load_into(g, wl)
        g.project(wl.dt, 3, TOL)
        ms = min(g.timeKernel(9, 300) for _ in range(8))
        g.destroy()
        return ms
    flat, square = fastest(100000, 16), fastest(1265, 1265)
    assert flat < 2.0 * square, (flat, square)
