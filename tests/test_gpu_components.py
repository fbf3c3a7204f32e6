"""Face weights of grids of one to many components a phase (densities summed in the weights' launch, and in one of their
own from thirteen components and 1024 tiles on), at odd and even counts and around tile edges: bit for bit the
FP64 oracle's.  More components cost their loads, not a memory latency each."""
import time

import numpy as np
import pytest

from fluidsim_amd import Context, FluidGridHIP, FluidGridState, FluidMixture, MixtureComponent

pytestmark = pytest.mark.gpu


def grid(W, H, nl, ng, context=None):
    rng = np.random.default_rng(100 * nl + ng)
    f = np.clip(rng.uniform(-0.5, 1.5, W * H), 0.0, 1.0)
    lm = [100.0 / nl * f * rng.uniform(0.5, 1.5, W * H) for _ in range(nl)]
    gm = [0.1 / ng * (1.0 - f) * rng.uniform(0.5, 1.5, W * H) + 1e-3 for _ in range(ng)]
    g = FluidGridHIP(W, H, 0.5, context=context)
    g.configureMaterials([], FluidMixture([MixtureComponent(f"l{k}", 100.0) for k in range(nl)]),
                         FluidMixture([MixtureComponent(f"g{k}", 0.1) for k in range(ng)]))
    g.upload(FluidGridState(f, np.zeros((W + 1) * H), np.zeros(W * (H + 1)), np.zeros(0), lm, gm))
    return g, f, lm, gm


@pytest.mark.parametrize("W,H,nl,ng", [(1, 1, 1, 1), (63, 15, 1, 2), (64, 16, 3, 1), (65, 17, 4, 5), (130, 70, 12, 11),
                                       (2048, 520, 7, 6), (2050, 515, 1, 1), (66000, 3, 6, 7), (64, 16384, 2, 12)])
def test_face_weights_are_bitwise(oracle, W, H, nl, ng):
    g, f, lm, gm = grid(W, H, nl, ng)
    o = oracle.OracleGrid(W, H, 0.5)
    o.configure([100.0] * nl, [0.1] * ng)
    o.upload(f, np.zeros((W + 1) * H), np.zeros(W * (H + 1)), None, np.concatenate(lm), np.concatenate(gm))
    for got, want in zip(g.faceWeights(), o.face_weights()):
        assert np.array_equal(got, want)
    g.destroy()


def test_components_travel_together():
    """A capillary force (which forms the face weights first) with 8 + 8 components against one with 1 + 1."""
    ctx = Context(0)

    def fastest(n):
        g = grid(300, 200, n, n, context=ctx)[0]
        g.setSurfaceTension(0.01)
        g.snapshotSave()
        times = []
        for _ in range(60):
            g.snapshotRestore()   # the weights are stale again
            ctx.synchronize()
            t = time.perf_counter()
            g.applySurfaceTension(1e-3)
            ctx.synchronize()
            times.append(time.perf_counter() - t)
        g.destroy()
        return min(times)
    one, many = fastest(1), fastest(8)
    ctx.close()
    assert many < 1.15 * one, (one, many)
