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
