"""The in-place FFT passes against FP64, over every radix and number of stages,
rows and columns that do not fill a tile, batches of grids and of frames, and
both signs; and the sizes beyond them, which rocFFT transforms."""
import numpy as np
import pytest

from fastrecon_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


# each axis: at most 6 stages of relative error below 3 units of 2^-24
@pytest.mark.parametrize("dim,N,C,F,sign", [
    (2, 2, 2, 0, 1), (2, 8, 3, 0, 1), (2, 9, 3, 0, 1), (2, 14, 2, 0, -1), (2, 16, 1, 0, 1), (2, 36, 1, 0, 1),
    (2, 49, 2, 0, 1), (2, 60, 5, 0, -1), (2, 96, 1, 0, 1), (2, 120, 3, 4, 1), (2, 126, 2, 0, 1), (2, 128, 1, 7, -1),
    (2, 162, 1, 0, 1), (2, 202, 2, 0, 1), (2, 243, 1, 0, 1), (2, 250, 2, 0, 1), (2, 256, 9, 0, 1), (2, 343, 1, 0, 1),
    (2, 384, 3, 0, -1), (2, 486, 1, 0, 1), (2, 500, 1, 3, 1), (2, 512, 8, 0, 1), (2, 640, 2, 0, 1), (2, 768, 1, 0, 1),
    (2, 1000, 1, 0, 1), (2, 1024, 1, 0, 1), (3, 10, 2, 0, 1), (3, 12, 3, 0, 1), (3, 21, 2, 0, -1), (3, 40, 5, 0, 1),
    (3, 60, 2, 0, 1), (3, 70, 1, 0, 1), (3, 90, 1, 0, 1), (3, 108, 2, 0, 1), (3, 128, 1, 0, 1)])
def test_transform(ctx, dim, N, C, F, sign):
    rng = np.random.default_rng(N * dim)
    n = max(F, 1) * N ** dim
    y = (rng.standard_normal((C, n)) + 1j * rng.standard_normal((C, n))).astype(np.complex64)
    g = hip.Grids(ctx, dim, N, C, frames=F)
    for c in range(C):
        g.upload(c, y[c])
    hip.FFT(ctx, dim, N, C * max(F, 1), sign)(g)
    axes = tuple(range(2, 2 + dim))
    z = y.reshape((C, max(F, 1)) + (N,) * dim).astype(np.complex128)
    ref = np.fft.ifftn(z, axes=axes) * N ** dim if sign > 0 else np.fft.fftn(z, axes=axes)
    for c in range(C):
        got = g.download(c).reshape(ref[c].shape)
        err = np.linalg.norm(got - ref[c]) / np.linalg.norm(ref[c])
        assert err <= dim * 6 * 3 * 2.0 ** -24


@pytest.mark.parametrize("dim,N,C,rc,shift,deapod", [
    (2, 96, 1, (48, 48, 1), True, False), (2, 90, 1, (37, 90, 1), True, True), (2, 45, 1, (45, 3, 1), False, True),
    (2, 100, 3, (50, 50, 1), True, False), (2, 512, 1, (250, 11, 1), True, True), (3, 70, 2, (35, 34, 1), True, True),
    (3, 64, 3, (64, 64, 64), True, False), (3, 66, 1, (33, 66, 20), False, False), (3, 20, 4, (10, 10, 10), True, True),
    (3, 75, 2, (30, 31, 75), False, True)])
def test_image_from_the_last_pass(ctx, dim, N, C, rc, shift, deapod):
    """The image and the grids, bitwise those of the transform and then the sum of squares."""
    rng = np.random.default_rng(N)
    y = (rng.standard_normal((C, N ** dim)) + 1j * rng.standard_normal((C, N ** dim))).astype(np.complex64)
    n = rc[0] * rc[1] * (rc[2] if dim == 3 else 1)
    dp = None
    if deapod:
        dp = hip.DeviceBuffer(ctx, 4 * n)
        dp.from_host(rng.uniform(0.5, 2.0, n).astype(np.float32))
    got = []
    for one in (True, False):
        g = hip.Grids(ctx, dim, N, C)
        f = hip.FFT(ctx, dim, N, C, +1)
        for c in range(C):
            g.upload(c, y[c])
        if one:
            out = hip.fft_sos(f, g, rc, shift, dp)
        else:
            f(g)
            out = hip.sos(ctx, g, rc, shift, dp)
        got.append((out.to_host(np.float32), np.stack([g.download(c) for c in range(C)])))
    np.testing.assert_array_equal(got[0][0].view(np.int32), got[1][0].view(np.int32))
    np.testing.assert_array_equal(got[0][1].view(np.int32), got[1][1].view(np.int32))
