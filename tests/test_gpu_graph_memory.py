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


def test_larger_crop_after_the_capture(ctx):
    N, C, rc, large = 256, 3, (64, 64, 1), (256, 200, 1)
    rng = np.random.default_rng(0)
    y = (rng.standard_normal((C, N * N)) + 1j * rng.standard_normal((C, N * N))).astype(np.complex64)
    t = rng.uniform(0, N - 1, (2000, 2)).astype(np.float32)
    s = hip.Samples(ctx, 2, 2000, C)
    s.set_traj(t)
    s.set_dcf(np.ones(2000, np.float32))
    s.set_coils(y[:, :2000])
    g, f = hip.Grids(ctx, 2, N, C), hip.FFT(ctx, 2, N, C)
    plan = hip.Plan(ctx, s, N, 4.0, hip.kb_lut(4.0, 2.0, 512)[0])
    out = hip.DeviceBuffer(ctx, 4 * rc[0] * rc[1])
    graph = hip.Graph(plan, s, g, f, rc, True, None, out)
    graph.launch()
    ref = out.to_host(np.int32)
    g2 = hip.Grids(ctx, 2, N, C)
    for c in range(C):
        g2.upload(c, y[c])
    wide = hip.fft_sos(f, g2, large).to_host(np.int32)
    size = 8 * C * rc[0] * N                                         # of the first pass' buffer
    held = [hip.DeviceBuffer(ctx, size) for _ in range(64)]
    mark = rng.integers(0, 255, size).astype(np.uint8)
    for b in held:
        b.from_host(mark)
    for turn in range(3):
        out.from_host(np.zeros(rc[0] * rc[1], np.float32))
        graph.launch()
        np.testing.assert_array_equal(out.to_host(np.int32), ref)
        for b in held:
            np.testing.assert_array_equal(b.to_host(np.uint8), mark)
        np.testing.assert_array_equal(hip.fft_sos(f, g2, large).to_host(np.int32), wide)
