"""Graphs whose passes hold scratch memory that a later, larger pass outgrows: every replay gives the eager result,
and leaves memory that was handed out since alone."""
import numpy as np
import pytest

from fastrecon_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


def scan(ctx, N, M, C, seed, tune=None):
    rng = np.random.default_rng(seed)
    t = rng.normal(N / 2, 2.0, (M, 3)).astype(np.float32)            # heavy boxes: partial sums
    y = (rng.standard_normal((C, M)) + 1j * rng.standard_normal((C, M))).astype(np.complex64)
    s = hip.Samples(ctx, 3, M, C)
    s.set_traj(t)
    s.set_dcf(np.ones(M, np.float32))
    s.set_coils(y)
    lut, _ = hip.kb_lut(4.0, 2.0, 512)
    return s, hip.Grids(ctx, 3, N, C), lut, y, t


@pytest.mark.parametrize("tune", [{}, dict(accumulate=5)])
def test_more_coils_after_the_capture(ctx, tune):
    N, M = 32, 20000
    s, g, lut, y, t = scan(ctx, N, M, 8, 0)
    plan = hip.Plan(ctx, s, N, 4.0, lut, dict(tune, split_taps=64))
    assert plan.info()["heavy_units"] > 0
    hip.grid_execute(plan, s, g)
    ref = g.download_all()
    graph = hip.Graph(plan, s, g)
    many = hip.Samples(ctx, 3, M, 72)                                # three chunks of coils instead of one
    many.set_traj(t)
    many.set_dcf(np.ones(M, np.float32))
    many.set_coils(np.resize(y, (72, M)))
    gm = hip.Grids(ctx, 3, N, 72)
    hip.grid_execute(plan, many, gm)
    others = []
    for seed in range(1, 5):                                         # plans from the memory that is free now
        so, go, _, _, _ = scan(ctx, N, M, 8, seed)
        po = hip.Plan(ctx, so, N, 4.0, lut, dict(tune, split_taps=64))
        hip.grid_execute(po, so, go)
        others.append((po, so, go, go.download_all()))
    for turn in range(3):
        g.upload(0, np.zeros(N ** 3, np.complex64))
        graph.launch()
        np.testing.assert_array_equal(g.download_all(), ref)
        for po, so, go, before in others:
            hip.grid_execute(po, so, go)
            np.testing.assert_array_equal(go.download_all(), before)
    np.testing.assert_array_equal(gm.download(0), ref[0])
