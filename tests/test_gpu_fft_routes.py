"""Transforms of sizes that few or many elements take to one implementation or the other: FP64 on both sides of the
lines between them, and one handle's grids as several of one grid each give them."""
import numpy as np
import pytest

from fastrecon_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


# each axis: at most 6 stages of relative error below 3 units of 2^-24, as for the other transforms
@pytest.mark.parametrize("dim,N,C,F,sign", [
    (2, 16, 3, 0, 1), (2, 48, 2, 60, -1), (2, 60, 2, 0, 1), (2, 60, 90, 0, 1), (2, 72, 10, 60, 1), (2, 96, 1, 0, 1),
    (2, 98, 60, 0, 1), (2, 98, 8, 16, 1), (2, 128, 27, 0, 1), (2, 128, 28, 0, -1), (2, 162, 8, 0, 1), (2, 162, 13, 0, 1),
    (2, 240, 4, 0, 1), (2, 240, 7, 0, 1), (2, 256, 6, 0, 1), (2, 256, 7, 0, 1), (2, 512, 1, 0, 1), (2, 512, 2, 0, 1),
    (3, 32, 2, 0, 1), (3, 32, 14, 0, 1), (3, 64, 3, 0, -1), (3, 64, 4, 0, -1), (3, 72, 1, 0, 1), (3, 72, 2, 0, 1),
    (3, 72, 5, 0, 1), (3, 112, 1, 0, 1), (3, 112, 2, 0, 1)])
def test_transform(ctx, dim, N, C, F, sign):
    rng = np.random.default_rng(N * dim + C)
    n = max(F, 1) * N ** dim
    g, one = hip.Grids(ctx, dim, N, C, frames=F), hip.Grids(ctx, dim, N, 1, frames=F)
    f, f1 = hip.FFT(ctx, dim, N, C * max(F, 1), sign), hip.FFT(ctx, dim, N, max(F, 1), sign)
    y = {}
    for c in range(C):
        v = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)
        g.upload(c, v)
        if c in (0, C - 1):
            y[c] = v
    f(g)
    axes = tuple(range(1, 1 + dim))
    for c, v in y.items():
        z = v.reshape((max(F, 1),) + (N,) * dim).astype(np.complex128)
        ref = np.fft.ifftn(z, axes=axes) * N ** dim if sign > 0 else np.fft.fftn(z, axes=axes)
        one.upload(0, v)
        f1(one)
        for got in (g.download(c), one.download(0)):
            err = np.linalg.norm(got.reshape(ref.shape) - ref) / np.linalg.norm(ref)
            assert err <= dim * 6 * 3 * 2.0 ** -24
