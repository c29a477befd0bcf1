"""Degridding and the density iterations on samples in tile order (the path
that a position-weight plan takes for kernels of width <= 4): bitwise against
the FP32 degrid oracle, and Pipe-Menon against the FP64 oracle.

Positions cover the edges of tiles and of the grid, points off the grid and
not finite, and more samples in one tile than one work item takes."""
import numpy as np
import pytest

from fastrecon_amd import hip

pytestmark = pytest.mark.gpu
SLICE = 1024            # samples per work item


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


def points(rng, dim, N, M):
    """Uniform points past both edges, a dense cluster, points on and next to
    cell and tile borders, and a few off the grid or not finite."""
    t = rng.uniform(-3.0, N + 2.0, (M, dim))
    t[: M // 3] = rng.normal(N / 2, 1.5, (M // 3, dim))
    k = M // 8
    t[M // 3: M // 3 + k] = rng.integers(0, N, (k, dim)) + rng.choice([0.0, 1e-6, -1e-6, 0.5], (k, dim))
    t = t.astype(np.float32)
    t[-1] = np.nan
    t[-2, 0] = np.inf
    t[-3, 0] = -np.inf
    t[-4] = 1e12
    return t


def build(ctx, t, N, C, width, frames=0, seed=0):
    M, dim = t.shape
    sizes = None
    if frames:
        sizes = np.full(frames, M // frames, np.int64)
        sizes[-1] += M - sizes.sum()
    s = hip.Samples(ctx, dim, M, C, frame_samples=sizes)
    s.set_traj(t)
    s.set_dcf(np.ones(M, np.float32))
    lut, _ = hip.kb_lut(width, 2.0, 512)
    return s, hip.Plan(ctx, s, N, width, lut), lut, sizes


@pytest.mark.parametrize("dim,N,M,C,width", [(3, 8, 2500, 1, 4.0), (3, 19, 5 * SLICE + 3, 2, 4.0), (3, 24, 4000, 3, 3.0),
                                             (3, 33, 3000, 4, 2.5), (3, 16, 2000, 9, 4.0), (2, 16, 700, 1, 4.0),
                                             (2, 37, 4 * SLICE + 1, 5, 4.0), (2, 50, 3000, 6, 1.0),
                                             (2, 64, 2000, 8, 3.7), (2, 20, 1500, 17, 4.0)])
def test_degrid_in_tile_order_is_bitwise(ctx, orc, dim, N, M, C, width):
    rng = np.random.default_rng(N + C)
    t = points(rng, dim, N, M)
    s, p, lut, _ = build(ctx, t, N, C, width)
    g = hip.Grids(ctx, dim, N, C)
    y = (rng.standard_normal((C, N ** dim)) + 1j * rng.standard_normal((C, N ** dim))).astype(np.complex64)
    out = hip.DeviceBuffer(ctx, 8 * M * C)
    hip.pipe_menon(p, s, 1, True)                # the plan now holds its tile order
    for bad in (False, True):
        if bad:                                  # only the samples that tap these cells see them
            y[0, (N ** dim) // 2] = np.inf
            y[-1, 0] = np.nan
        for c in range(C):
            g.upload(c, y[c])
        hip.degrid_execute(p, s, g, out)
        got = np.ascontiguousarray(out.to_host(np.complex64).reshape(M, C).T)
        ref = orc.degrid_f32(t, y, N, width, lut)
        if bad:
            a, b = got.view(np.float32), ref.view(np.float32)
            assert np.array_equal(np.isnan(a), np.isnan(b))
            ok = ~np.isnan(b)
            assert not ok.all()
            assert np.array_equal(a[ok], b[ok])
        else:
            np.testing.assert_array_equal(got.view(np.int32), ref.view(np.int32))


def test_degrid_of_frames_in_tile_order(ctx, orc):
    rng = np.random.default_rng(2)
    N, C, F, M = 40, 3, 5, 3600
    t = points(rng, 2, N, M)
    s, p, lut, sizes = build(ctx, t, N, C, 4.0, F)
    g = hip.Grids(ctx, 2, N, C, frames=F)
    y = (rng.standard_normal((C, F * N * N)) + 1j * rng.standard_normal((C, F * N * N))).astype(np.complex64)
    for c in range(C):
        g.upload(c, y[c])
    out = hip.DeviceBuffer(ctx, 8 * M * C)
    hip.pipe_menon(p, s, 1, True)
    hip.degrid_execute(p, s, g, out)
    got = np.ascontiguousarray(out.to_host(np.complex64).reshape(M, C).T)
    o = 0
    for f, n in enumerate(sizes):
        ref = orc.degrid_f32(t[o:o + n], np.ascontiguousarray(y[:, f * N * N:(f + 1) * N * N]), N, 4.0, lut)
        np.testing.assert_array_equal(np.ascontiguousarray(got[:, o:o + n]).view(np.int32), ref.view(np.int32))
        o += n


def test_degrid_follows_a_changed_trajectory(ctx, orc):
    """A handle whose trajectory is not the plan's degrids at its own points."""
    rng = np.random.default_rng(3)
    N, M = 24, 2000
    t = rng.uniform(0, N - 1, (M, 3)).astype(np.float32)
    s, p, lut, _ = build(ctx, t, N, 1, 4.0)
    hip.pipe_menon(p, s, 1, True)
    g = hip.Grids(ctx, 3, N, 1)
    y = (rng.standard_normal((1, N ** 3)) + 1j * rng.standard_normal((1, N ** 3))).astype(np.complex64)
    g.upload(0, y[0])
    out = hip.DeviceBuffer(ctx, 8 * M)
    t2 = rng.uniform(0, N - 1, (M, 3)).astype(np.float32)
    s.set_traj(t2)
    hip.degrid_execute(p, s, g, out)
    ref = orc.degrid_f32(t2, y, N, 4.0, lut)
    np.testing.assert_array_equal(out.to_host(np.complex64).view(np.int32), ref.view(np.int32).ravel())


@pytest.mark.parametrize("dim,N,M,width,ones", [(3, 8, 400, 4.0, True), (3, 27, 20 * SLICE + 7, 4.0, True),
                                                (3, 32, 9000, 3.0, False), (2, 16, 300, 4.0, False),
                                                (2, 53, 30 * SLICE, 4.0, True), (2, 90, 20000, 2.0, True)])
def test_pipe_menon_in_tile_order(ctx, orc, dim, N, M, width, ones):
    """Against the FP64 oracle, from ones or from the handle's density, twice
    the same bits.  Bar: 1e-6 as for the other Pipe-Menon tests (FP32 sums
    and ratios, a few roundings of 6e-8 per iteration)."""
    rng = np.random.default_rng(N)
    t = rng.uniform(-1.0, N, (M, dim))
    t[: M // 2] = rng.normal(N / 2, N / 12, (M // 2, dim))
    t = t.astype(np.float32)
    s, p, lut, _ = build(ctx, t, N, 1, width)
    got = []
    for _ in range(2):
        s.set_dcf(np.ones(M, np.float32))
        hip.pipe_menon(p, s, 6, ones)
        got.append(s.get_dcf())
    assert np.array_equal(got[0], got[1])
    ref = orc.pipe_menon(t, N, width, lut, iters=6)
    e = np.linalg.norm(got[0] - ref) / np.linalg.norm(ref)
    print(f"[pipe-menon dim={dim} N={N} M={M}] rel-L2 {e:.2e}", flush=True)
    assert e <= 1e-6
