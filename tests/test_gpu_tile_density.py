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


@pytest.mark.parametrize("dim,N,M", [(3, 27, 6000), (2, 53, 9000)])
def test_start_from_a_density(ctx, orc, dim, N, M):
    """Three iterations and three more from their density are six, bit for bit; from a random density, the FP64
    oracle's (bar: 1e-6 as for the other Pipe-Menon tests)."""
    rng = np.random.default_rng(N)
    t = rng.uniform(-1.0, N, (M, dim))
    t[: M // 2] = rng.normal(N / 2, N / 12, (M // 2, dim))
    t = t.astype(np.float32)
    lut, _ = hip.kb_lut(4.0, 2.0, 512)
    s = samples(ctx, t, np.ones(M, np.float32))
    p = hip.Plan(ctx, s, N, 4.0, lut)
    hip.pipe_menon(p, s, 6, True)
    six = s.get_dcf()
    hip.pipe_menon(p, s, 3, True)
    hip.pipe_menon(p, s, 3, False)
    np.testing.assert_array_equal(s.get_dcf().view(np.int32), six.view(np.int32))
    w0 = rng.uniform(0.1, 3.0, M).astype(np.float32)
    s.set_dcf(w0)
    hip.pipe_menon(p, s, 4, False)
    ref = orc.pipe_menon(t, N, 4.0, lut, iters=4, w0=w0)
    e = np.linalg.norm(s.get_dcf() - ref) / np.linalg.norm(ref)
    print(f"[pipe-menon from a density dim={dim} N={N}] rel-L2 {e:.2e}", flush=True)
    assert e <= 1e-6
