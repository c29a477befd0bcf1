"""Position-weight plans at the limits of their record counts."""
import numpy as np
import pytest

from fastrecon_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


def unit_table_plan(ctx, t, y, N, width, tune=None):
    """A plan whose weights are all 1 inside the kernel, and its samples."""
    M, dim = t.shape
    s = hip.Samples(ctx, dim, M, 1)
    s.set_traj(t)
    s.set_dcf(np.ones(M, np.float32))
    s.set_coil(0, y)
    return s, hip.Plan(ctx, s, N, width, np.ones(64, np.float32), tune)


def test_more_than_2_30_records(ctx):
    """Records beyond 4 GiB: the grid of all samples is the sum of the grids of their halves, exactly (unit weights
    and small whole numbers: no cell's sum reaches 2^24)."""
    rng = np.random.default_rng(0)
    N, M, width = 64, 7_000_000, 16.0
    t = rng.uniform(0, N - 1, (M, 3)).astype(np.float32)
    y = rng.integers(0, 3, M).astype(np.complex64)
    grids = []
    for part in (slice(0, M), slice(0, M // 2), slice(M // 2, M)):
        s, p = unit_table_plan(ctx, t[part], y[part], N, width)
        records = p.info()["records"]
        assert (records > 1 << 30) == (part == slice(0, M)), records
        g = hip.Grids(ctx, 3, N, 1)
        hip.grid_execute(p, s, g)
        grids.append(g.download(0))
        for h in (g, p, s):
            h.close()
    assert grids[0].real.max() < 1 << 24
    np.testing.assert_array_equal(grids[0], grids[1] + grids[2])


def corner(ctx, N, shift, M):
    """Records of a plan, and the gridded and degridded samples, of points within 64^3 cells from `shift` on."""
    rng = np.random.default_rng(1)
    t = (rng.integers(4 * 64, 60 * 64, (M, 3)) / 64).astype(np.float32)
    s = hip.Samples(ctx, 3, M, 1)
    s.set_traj(t + np.float32(shift))
    s.set_dcf(np.ones(M, np.float32))
    s.set_coil(0, rng.standard_normal((M, 2)).astype(np.float32).view(np.complex64)[:, 0])
    p = hip.Plan(ctx, s, N, 4.0, hip.kb_lut(4.0, 2.0, 512)[0])
    g = hip.Grids(ctx, 3, N, 1)
    out = hip.DeviceBuffer(ctx, 8 * M)
    hip.grid_execute(p, s, g)
    hip.degrid_execute(p, s, g, out)
    got = p.info()["records"], out.to_host(np.int32)
    for h in (out, g, p, s):
        h.close()
    return got


def test_more_boxes_than_records(ctx):
    """The records are refused by what they take when padded, and boxes without any take nothing.  Weights and sums
    are those of the same samples on a small grid, bit for bit (shifts are multiples of the unit boxes' sides)."""
    N, M = 1288, 1_700_000
    small, large = corner(ctx, 64, 0, M), corner(ctx, N, 1220, M)
    assert small[0] == large[0]
    assert small[0] + 16 * (N // 4) * (N // 2) ** 2 >= 1 << 31
    np.testing.assert_array_equal(small[1], large[1])


def test_more_units_than_a_launch_has_waves(ctx):
    """1290^3 does not divide into pairs of boxes: 134M units, of which a launch takes 67M at one a wave."""
    M = 3000
    small, large = corner(ctx, 64, 0, M), corner(ctx, 1290, 1220, M)
    assert small[0] == large[0]
    np.testing.assert_array_equal(small[1], large[1])


def test_data_past_4_gib(ctx):
    """Rows addressed in 64 bits: coils of one data set times powers of two, bit for bit that set's grid times them."""
    rng = np.random.default_rng(2)
    N, M, C = 48, 8_400_000, 65
    t = rng.uniform(0, N - 1, (M, 3)).astype(np.float32)
    y = rng.standard_normal((M, 2)).astype(np.float32).view(np.complex64)[:, 0]
    lut, _ = hip.kb_lut(4.0, 2.0, 512)
    grids = []
    for coils in (1, C):
        s = hip.Samples(ctx, 3, M, coils)
        assert (8 * (M + 1) * coils >= 1 << 32) == (coils == C)
        s.set_traj(t)
        s.set_dcf(np.ones(M, np.float32))
        for c in range(coils):
            s.set_coil(c, y * np.float32(2.0 ** (c % 7)))
        g = hip.Grids(ctx, 3, N, coils)
        p = hip.Plan(ctx, s, N, 4.0, lut)
        hip.grid_execute(p, s, g)
        grids.append(g.download_all())
        for h in (g, p, s):
            h.close()
    for c in range(C):
        np.testing.assert_array_equal(grids[1][c], grids[0][0] * np.float32(2.0 ** (c % 7)))


def test_degridding_of_2_32_values(ctx):
    """More sample-coils than a launch has work-items along one axis, by the general kernel (a wide kernel)."""
    rng = np.random.default_rng(3)
    N, M, C, width, part = 16, 1 << 26, 66, 4.5, 1000
    t = rng.integers(0, 16 * (N - 1), (part, 3)).astype(np.float32) / 16
    all_t = np.empty((M, 3), np.float32)
    all_t[:] = t[0]
    all_t[:part] = all_t[-part:] = t
    lut, _ = hip.kb_lut(width, 2.0, 64)
    g = hip.Grids(ctx, 3, N, C)
    for c in range(C):
        g.upload(c, (rng.standard_normal(N ** 3) + 1j * rng.standard_normal(N ** 3)).astype(np.complex64))

    def handle(points):
        s = hip.Samples(ctx, 3, len(points), 1)
        s.set_traj(points)
        return s

    s = handle(t)
    small = hip.DeviceBuffer(ctx, 8 * part * C)
    hip.degrid_execute(hip.Plan(ctx, s, N, width, lut, dict(accumulate=2)), s, g, small)
    ref = small.to_host(np.int32)
    s = handle(all_t)
    plan = hip.Plan(ctx, s, N, width, lut)
    out = hip.DeviceBuffer(ctx, 8 * M * C)
    last = hip.DevicePtr(out, 8 * C * (M - part))
    zero = np.zeros(2 * part * C, np.float32)
    got = np.empty(2 * part * C, np.int32)
    L = ctx.L
    for p in (out.ptr, last.ptr):
        ctx.check(L.fr_memcpy_h2d(ctx.h, p, zero.ctypes.data, zero.nbytes), "fr_memcpy_h2d")
    hip.degrid_execute(plan, s, g, out)
    for p in (out.ptr, last.ptr):
        ctx.check(L.fr_memcpy_d2h(ctx.h, got.ctypes.data, p, got.nbytes), "fr_memcpy_d2h")
        np.testing.assert_array_equal(got, ref)
    for h in (out, plan, s, g):
        h.close()
