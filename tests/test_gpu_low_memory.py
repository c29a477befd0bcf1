"""Degridding and Pipe-Menon where the device has no memory for the samples' tile order: the general kernels, which
need less, still answer."""
import numpy as np
import pytest

from fastrecon_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


class little_left:
    """Takes the device's memory but for about `left` bytes."""

    def __init__(self, ctx, left):
        self.ctx, self.left = ctx, left

    def __enter__(self):
        keep, self.taken = hip.DeviceBuffer(self.ctx, self.left), []
        for size in (1 << 36, 1 << 33, 1 << 30, 1 << 27, 1 << 25):
            try:
                while len(self.taken) < 4000:
                    self.taken.append(hip.DeviceBuffer(self.ctx, size))
            except hip.HipError:
                pass
        keep.close()

    def __exit__(self, *error):
        for b in self.taken:
            b.close()


def test_degridding(ctx):
    rng = np.random.default_rng(0)
    N, M = 256, 24_000_000
    t = rng.random((M, 2), np.float32) * np.float32(N - 1)
    s = hip.Samples(ctx, 2, M, 1)
    s.set_traj(t)
    lut, _ = hip.kb_lut(1.5, 2.0, 64)
    p = hip.Plan(ctx, s, N, 1.5, lut)
    g = hip.Grids(ctx, 2, N, 1)
    g.upload(0, (rng.standard_normal(N * N) + 1j * rng.standard_normal(N * N)).astype(np.complex64))
    out = hip.DeviceBuffer(ctx, 8 * M)
    hip.degrid_execute(hip.Plan(ctx, s, N, 1.5, lut, dict(accumulate=5)), s, g, out)     # the general kernel
    ref = out.to_host(np.int32)
    with little_left(ctx, 200 << 20):                # the sorted positions alone take 384 MB
        hip.degrid_execute(p, s, g, out)
    np.testing.assert_array_equal(out.to_host(np.int32), ref)
    hip.degrid_execute(p, s, g, out)                 # in tile order, once there is memory
    np.testing.assert_array_equal(out.to_host(np.int32), ref)


def test_pipe_menon(ctx):
    rng = np.random.default_rng(1)
    N, M = 512, 1_000_000
    t = rng.random((M, 3), np.float32) * np.float32(N - 1)
    s = hip.Samples(ctx, 3, M, 1)
    s.set_traj(t)
    s.set_dcf(np.ones(M, np.float32))
    lut, _ = hip.kb_lut(4.0, 2.0, 512)
    p = hip.Plan(ctx, s, N, 4.0, lut)
    with little_left(ctx, 1600 << 20):               # the general path takes 1.2 GB; the tiles' boxes alone 1.3 GB
        hip.pipe_menon(p, s, 3, True)
    low = s.get_dcf()
    hip.pipe_menon(p, s, 3, True)
    e = np.linalg.norm(low - s.get_dcf()) / np.linalg.norm(low)
    print(f"[pipe-menon] general against tile order rel-L2 {e:.2e}", flush=True)
    assert e <= 1e-6
