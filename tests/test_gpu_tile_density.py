"""Pipe-Menon on samples in tile order: densities that are not finite, and a start from the handle's own density."""
import numpy as np
import pytest

from fastrecon_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


def samples(ctx, t, dcf):
    s = hip.Samples(ctx, t.shape[1], t.shape[0], 1)
    s.set_traj(t)
    s.set_dcf(dcf)
    return s


@pytest.mark.parametrize("dim,N,M", [(3, 24, 3000), (3, 19, 2000), (2, 50, 1500), (2, 64, 4000)])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_density_that_is_not_finite(ctx, dim, N, M, value):
    """It reaches the samples that share a cell with it, and no others: the zeros are those of the sequential kernels
    (an exact-order plan), the others agree to 1e-5 (an infinite one over its infinite
    denominator is NaN in both)."""
    rng = np.random.default_rng(N)
    t = rng.uniform(-1.0, N, (M, dim)).astype(np.float32)
    w = np.ones(M, np.float32)
    w[rng.integers(0, M, 3)] = value
    lut, _ = hip.kb_lut(4.0, 2.0, 512)
    got = []
    for tune in (None, dict(exact_order=1)):
        s = samples(ctx, t, w)
        hip.pipe_menon(hip.Plan(ctx, s, N, 4.0, lut, tune), s, 1, False)
        got.append(s.get_dcf())
    assert 0 < (got[1] == 0).sum() < M // 2
    np.testing.assert_array_equal(got[0] == 0, got[1] == 0)
    np.testing.assert_allclose(got[0], got[1], rtol=1e-5)
