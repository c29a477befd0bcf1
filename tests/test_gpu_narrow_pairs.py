"""Unit boxes less than 4 cells wide, gridded in pairs: the bits of the same boxes written out one by one."""
import numpy as np
import pytest

from fastrecon_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("dim,N,box", [(3, 16, (2, 2, 4)), (3, 24, (2, 4, 2)), (3, 16, (1, 4, 4)), (3, 32, (1, 2, 8)),
                                       (3, 32, (2, 8, 1)), (2, 48, (2, 8, 1)), (2, 32, (1, 16, 1)), (3, 16, (4, 2, 2))])
@pytest.mark.parametrize("C,half", [(1, False), (8, False), (11, True), (16, False), (21, False), (34, True)])
def test_pairs_of_narrow_boxes(ctx, dim, N, box, C, half):
    rng = np.random.default_rng(N + C)
    M = 4000
    t = rng.uniform(-1.0, N, (M, dim))
    t[: M // 4] = rng.normal(N / 2, 0.7, (M // 4, dim))              # front units, whose partners go alone
    s = hip.Samples(ctx, dim, M, C, hip.FR_SAMPLES_C16 if half else hip.FR_SAMPLES_C64)
    s.set_traj(t.astype(np.float32))
    s.set_dcf(rng.uniform(0.5, 2.0, M).astype(np.float32))
    s.set_coils((rng.standard_normal((C, M)) + 1j * rng.standard_normal((C, M))).astype(np.complex64))
    lut, _ = hip.kb_lut(4.0, 2.0, 512)
    got = []
    for writes in (0, 2):
        p = hip.Plan(ctx, s, N, 4.0, lut, dict(tile_x=box[0], tile_y=box[1], tile_z=box[2], tile_writes=writes))
        g = hip.Grids(ctx, dim, N, C)
        hip.grid_execute(p, s, g)
        got.append(g.download_all())
    np.testing.assert_array_equal(got[0].view(np.int32), got[1].view(np.int32))


@pytest.mark.parametrize("dim,N,box", [(3, 64, (2, 2, 4)), (3, 64, (2, 4, 2)), (2, 512, (2, 8, 1)), (3, 64, (1, 4, 4))])
def test_narrow_boxes_come_in_pairs(ctx, dim, N, box):
    """The identity scale's sample of the grid is of pairs: with a stride it is an estimate, not the whole sum."""
    rng = np.random.default_rng(N)
    M = 20000                                                        # few records a box: most boxes are light
    t = rng.uniform(0, N - 1, (M, dim)).astype(np.float32)
    w = rng.uniform(0.1, 2.0, M).astype(np.float32)
    lut, _ = hip.kb_lut(4.0, 2.0, 512)
    alpha = []
    for stride in (1, 4):
        s = hip.Samples(ctx, dim, M, 1)
        s.set_traj(t)
        s.set_dcf(w)
        p = hip.Plan(ctx, s, N, 4.0, lut, dict(tile_x=box[0], tile_y=box[1], tile_z=box[2]))
        alpha.append(hip.dcf_identity_scale(p, s, stride))
    assert alpha[0] != alpha[1]
    assert abs(alpha[1] / alpha[0] - 1) < 0.2
