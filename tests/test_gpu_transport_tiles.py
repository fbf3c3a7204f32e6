"""Transport passes at the edges of their tiles (63 cells of a wavefront along x, 7 rows of a workgroup along y, 64 x 16
cells of the set-up), with one to three components a phase, one substep and several: bit for bit the FP64 oracle's, on
random fractions and velocities.  A refused call (more substeps than allowed, found out while the first one is already
queued) changes nothing."""
import numpy as np
import pytest

from fluidsim_amd import FluidGridHIP, FluidGridState, FluidMixture, MixtureComponent

pytestmark = pytest.mark.gpu


def state(W, H, nl, ng, seed):
    rng = np.random.default_rng(seed)
    f = np.clip(rng.uniform(-0.5, 1.5, W * H), 0.0, 1.0)
    u, v = rng.normal(size=(H, W + 1)), rng.normal(size=(H + 1, W))
    u[:, [0, W]] = 0.0
    v[[0, H], :] = 0.0
    lm = [100.0 / nl * f * rng.uniform(0.5, 1.5, W * H) for _ in range(nl)]
    gm = [0.1 / ng * (1.0 - f) * rng.uniform(0.5, 1.5, W * H) for _ in range(ng)]
    return f, u.ravel(), v.ravel(), lm, gm


def grid(W, H, s):
    f, u, v, lm, gm = s
    g = FluidGridHIP(W, H, 1.0)
    g.configureMaterials([], FluidMixture([MixtureComponent(f"l{k}", 100.0) for k in range(len(lm))]),
                         FluidMixture([MixtureComponent(f"g{k}", 0.1) for k in range(len(gm))]))
    g.upload(FluidGridState(f, u, v, np.zeros(0), lm, gm))
    return g


@pytest.mark.parametrize("W,H", [(1, 1), (1, 40), (40, 1), (62, 6), (63, 7), (64, 8), (65, 15), (126, 14), (127, 16),
                                 (130, 33)])
@pytest.mark.parametrize("nl,ng,dt", [(1, 1, 0.05), (2, 2, 0.6), (3, 1, 0.3)])
def test_transport_at_tile_edges_is_bitwise(oracle, W, H, nl, ng, dt):
    s = state(W, H, nl, ng, W * 1000 + H)
    g = grid(W, H, s)
    o = oracle.OracleGrid(W, H, 1.0)
    o.configure([100.0] * nl, [0.1] * ng)
    o.upload(s[0], s[1], s[2], None, np.concatenate(s[3]), np.concatenate(s[4]))
    assert g.advect(dt) == o.advect(dt)
    a, b = g.download(), o.download()
    g.destroy()
    for name, got in (("fraction", a.liquid_fraction), ("u", a.u), ("v", a.v),
                      ("liquid_mass", np.concatenate(a.liquid_mass)), ("gas_mass", np.concatenate(a.gas_mass))):
        assert np.array_equal(got, b[name], equal_nan=True), name


def test_a_refused_transport_changes_nothing():
    W, H = 70, 20
    f, u, v, lm, gm = state(W, H, 2, 2, 5)
    u[W + 5] = 1e9
    g = grid(W, H, (f, u, v, lm, gm))
    with pytest.raises(RuntimeError):
        g.advect(1.0)
    a = g.download()
    g.destroy()
    assert np.array_equal(a.liquid_fraction, f) and np.array_equal(a.u, u) and np.array_equal(a.v, v)
    assert np.array_equal(np.concatenate(a.liquid_mass), np.concatenate(lm))
    assert np.array_equal(np.concatenate(a.gas_mass), np.concatenate(gm))
