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
