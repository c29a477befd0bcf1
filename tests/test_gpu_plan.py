"""Position-weight plans: the (sample, unit box) records that the nearest-cell
test finds against the reference's tap test over every cell
(GridLut.cpp:99-136), and plans built in memory that earlier plans gave back."""
import itertools

import numpy as np
import pytest

from fastrecon_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


def points(rng, dim, N, M, width):
    """Points past both edges; on cells, half cells and at the kernel's
    half-width (and one ulp to either side) from box borders; not finite."""
    t = rng.uniform(-3.0, N + 2.0, (M, dim))
    k = M // 2
    at = rng.integers(-2, N + 2, (k, dim)) + rng.choice([0.0, 0.5, width / 2, -width / 2], (k, dim))
    at = at.astype(np.float32)
    step = rng.integers(0, 3, (k, dim))
    at = np.where(step == 1, np.nextafter(at, np.float32(1e9)), np.where(step == 2, np.nextafter(at, np.float32(-1e9)), at))
    t = t.astype(np.float32)
    t[:k] = at
    t[-1], t[-2, 0], t[-3, 0] = np.nan, np.inf, -np.inf
    return t


def records(t, N, width, box):
    """Pairs of sample and box with an accepted tap, by the reference's FP32 test of each cell."""
    hw = np.float32(width / 2)
    pairs = set()
    for i, c in enumerate(t):
        if not np.isfinite(c).all():
            continue
        axes = [np.arange(max(int(np.ceil(v - hw)), 0), min(int(np.floor(v + hw)), N - 1) + 1) for v in c]
        for cell in itertools.product(*axes[::-1]):
            d = [np.float32(x) - v for x, v in zip(cell, c[::-1])]          # z, y, x
            d2 = np.float32(0.0)
            for v in d:
                d2 = np.float32(d2 + np.float32(v * v))
            if np.sqrt(d2) < hw:
                pairs.add((i, tuple(x // b for x, b in zip(cell[::-1], box))))
    return len(pairs)


@pytest.mark.parametrize("dim,N,M,width", [(3, 8, 900, 4.0), (3, 13, 500, 3.0), (3, 6, 300, 7.5), (3, 32, 400, 1.0),
                                           (2, 16, 900, 4.0), (2, 21, 900, 2.5), (2, 2, 64, 4.0), (2, 64, 513, 16.0)])
def test_records(ctx, dim, N, M, width):
    t = points(np.random.default_rng(N), dim, N, M, width)
    s = hip.Samples(ctx, dim, M, 1)
    s.set_traj(t)
    lut, _ = hip.kb_lut(width, 2.0, 256)
    box = [min(b, N) for b in ((8, 2) if dim == 2 else (4, 2, 2))]
    assert hip.Plan(ctx, s, N, width, lut).info()["records"] == records(t, N, width, box)


def test_memory_given_back(ctx):
    """Grids of plans built one after the other, of other sizes in between."""
    lut, _ = hip.kb_lut(4.0, 2.0, 256)
    first = {}
    for turn in range(3):
        for N, M in ((32, 5000), (24, 40000), (31, 1), (40, 40000)):
            t = np.random.default_rng(N).uniform(0, N, (M, 3)).astype(np.float32)
            t[: M // 2] = np.random.default_rng(M).normal(N / 2, 0.5, (M // 2, 3))       # heavy boxes: partial sums
            y = np.random.default_rng(1).standard_normal((M, 4)).astype(np.float32).view(np.complex64)
            s = hip.Samples(ctx, 3, M, 2)
            s.set_traj(t)
            s.set_dcf(np.ones(M, np.float32))
            for c in range(2):
                s.set_coil(c, np.ascontiguousarray(y[:, c]))
            g = hip.Grids(ctx, 3, N, 2)
            hip.grid_execute(hip.Plan(ctx, s, N, 4.0, lut), s, g)
            got = np.stack([g.download(c) for c in range(2)])
            assert np.isfinite(got.view(np.float32)).all()
            np.testing.assert_array_equal(got, first.setdefault(N, got))
