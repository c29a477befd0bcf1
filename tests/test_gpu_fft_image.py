"""Images from the transforms: their distance from FP64, and the single-coil
image that the last pass forms."""
import numpy as np
import pytest
import scipy.fft

from fastrecon_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("N", [100, 180, 250, 288, 300])
def test_image_of_coils_is_as_exact_as_another_fp32_transform(ctx, N):
    """A sum of squares over coils averages the roundings of the elements, but not errors that all elements share
    (the roundings of a butterfly's constants).  Bar: the distance from FP64 of the same image by scipy's FP32
    transform."""
    C, h = 5, N // 4
    rng = np.random.default_rng(0)
    k = (np.arange(N) - (N - 1) / 2) / N
    rho = np.hypot(k[:, None], k[None, :])
    w = rng.standard_normal((C, N, N)) + 1j * rng.standard_normal((C, N, N))
    z = (w * (0.05 + 1 / (1 + 40 * rho)) * (rho < 0.5)).astype(np.complex64)     # an object's spectrum
    g = hip.Grids(ctx, 2, N, C)
    for c in range(C):
        g.upload(c, z[c].ravel())
    hip.FFT(ctx, 2, N, C, +1)(g)
    keep = np.ix_(np.r_[:h, N - h:N], np.r_[:h, N - h:N])

    def image(y):
        return np.sqrt(sum(np.abs(v[keep].astype(np.complex128)) ** 2 for v in y))

    ref = image(scipy.fft.ifftn(z.astype(np.complex128), axes=(1, 2), norm="forward"))

    def off(y):
        return np.linalg.norm(image(y) - ref) / np.linalg.norm(ref)

    got, other = off(g.download_all().reshape(C, N, N)), off(scipy.fft.ifftn(z, axes=(1, 2), norm="forward"))
    print(f"[image {N}^2 x {C}] {got:.3e}, scipy FP32 {other:.3e}", flush=True)
    assert got <= other


@pytest.mark.parametrize("dim,N,rc,shift,deapod", [
    (3, 12, (12, 12, 12), True, False), (3, 20, (10, 7, 20), True, True), (3, 45, (17, 45, 1), False, True),
    (3, 64, (64, 31, 40), True, True), (3, 70, (1, 35, 66), True, False), (3, 63, (30, 31, 32), False, False),
    (3, 100, (50, 49, 47), True, True), (3, 105, (105, 53, 20), False, True), (3, 120, (60, 61, 62), True, True),
    (2, 96, (47, 96, 1), True, True), (2, 90, (90, 1, 1), False, False), (2, 1000, (500, 333, 1), True, True)])
def test_single_coil(ctx, dim, N, rc, shift, deapod):
    """The image of fr_fft_sos and the transformed grid, bitwise those of the transform and then the sum of squares,
    up to and past the size from which they are formed apart."""
    rng = np.random.default_rng(N)
    y = (rng.standard_normal(N ** dim) + 1j * rng.standard_normal(N ** dim)).astype(np.complex64)
    n = rc[0] * rc[1] * (rc[2] if dim == 3 else 1)
    dp = None
    if deapod:
        dp = hip.DeviceBuffer(ctx, 4 * n)
        dp.from_host(rng.uniform(0.5, 2.0, n).astype(np.float32))
    got = []
    for one in (True, False):
        g, f = hip.Grids(ctx, dim, N, 1), hip.FFT(ctx, dim, N, 1, +1)
        g.upload(0, y)
        if one:
            out = hip.fft_sos(f, g, rc, shift, dp)
        else:
            f(g)
            out = hip.sos(ctx, g, rc, shift, dp)
        got.append((out.to_host(np.int32), g.download(0).view(np.int32)))
    np.testing.assert_array_equal(got[0][0], got[1][0])
    np.testing.assert_array_equal(got[0][1], got[1][1])
