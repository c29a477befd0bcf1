"""Cropped FFT + sum of squares of a single 2D image, whose passes split the
work over more workgroups than those of many images: bitwise the sums of the
passes that batches of frames take."""
import numpy as np
import pytest

from fastrecon_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


def image(ctx, y, N, rc, deapod):
    C, F = y.shape[:2]
    g = hip.Grids(ctx, 2, N, C, frames=F)
    for c in range(C):
        g.upload(c, np.ascontiguousarray(y[c].reshape(-1)))
    out = hip.DeviceBuffer(ctx, 4 * F * rc[0] * rc[1])
    hip.fft_sos(hip.FFT(ctx, 2, N, C * F, +1), g, (rc[0], rc[1], 1), True, deapod, out)
    return out.to_host(np.float32).reshape(F, -1)


@pytest.mark.parametrize("N,rc,C", [(512, (256, 256), 8), (512, (512, 512), 1), (512, (16, 1), 2), (512, (304, 511), 3),
                                    (384, (192, 192), 5), (384, (16, 384), 4), (256, (128, 128), 9),
                                    (256, (256, 256), 17), (256, (48, 7), 32)])
def test_single_images_as_frames(ctx, N, rc, C):
    rng = np.random.default_rng(N + C)
    F = -(-600 * 8 // rc[0])                     # enough frames for the passes of many images
    few = 3
    y = (rng.standard_normal((C, few, N * N)) + 1j * rng.standard_normal((C, few, N * N))).astype(np.complex64)
    d = hip.DeviceBuffer(ctx, 4 * rc[0] * rc[1])
    d.from_host(rng.uniform(0.5, 2.0, rc[0] * rc[1]).astype(np.float32))
    one = np.concatenate([image(ctx, y[:, f:f + 1], N, rc, d) for f in range(few)])
    ref = np.abs(np.fft.ifft2(y[:, 0].reshape(C, N, N).astype(np.complex128)) * N * N)
    x0, y0 = (N - rc[0]) // 2, (N - rc[1]) // 2
    ref = np.fft.fftshift(ref, axes=(1, 2))[:, y0:y0 + rc[1], x0:x0 + rc[0]]
    ref = np.sqrt((ref ** 2).sum(0)).reshape(-1) / d.to_host(np.float32)
    assert np.abs(one[0] - ref).max() <= 1e-5 * ref.max()
    if C * F * N * N * 8 > 2 << 30:
        F = max(few, (2 << 30) // (C * N * N * 8))
    many = np.zeros((C, F, N * N), np.complex64)
    many[:, :few] = y
    np.testing.assert_array_equal(image(ctx, many, N, rc, d)[:few].view(np.int32), one.view(np.int32))
