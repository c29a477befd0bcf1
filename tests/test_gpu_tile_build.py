"""The samples' tile order that the first large degridding builds, and its absence under capture."""
import ctypes as C

import numpy as np
import pytest

from fastrecon_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


class Capture:
    """What is enqueued on the context's stream inside the block, as a graph."""

    def __init__(self, ctx):
        self.hip, self.stream = C.CDLL("libamdhip64.so"), C.c_void_p(ctx.stream)
        self.graph, self.exec = C.c_void_p(), C.c_void_p()

    def __enter__(self):
        assert self.hip.hipStreamBeginCapture(self.stream, 1) == 0
        return self

    def __exit__(self, *error):
        assert self.hip.hipStreamEndCapture(self.stream, C.byref(self.graph)) == 0
        assert self.hip.hipGraphInstantiate(C.byref(self.exec), self.graph, None, None, C.c_size_t(0)) == 0

    def launch(self):
        assert self.hip.hipGraphLaunch(self.exec, self.stream) == 0

    def close(self):
        self.hip.hipGraphExecDestroy(self.exec)
        self.hip.hipGraphDestroy(self.graph)


@pytest.mark.parametrize("dim,N,M,coils", [(3, 40, (1 << 21) + 5, 4), (2, 100, (1 << 20) + 3, 9)])
def test_first_large_degridding(ctx, dim, N, M, coils):
    """On a fresh plan, captured and then eager: the bits of the general kernel (an equal trajectory in another
    handle), at every replay."""
    rng = np.random.default_rng(N)
    t = rng.uniform(-2.0, N + 1.0, (M, dim)).astype(np.float32)
    lut, _ = hip.kb_lut(4.0, 2.0, 512)
    g = hip.Grids(ctx, dim, N, coils)
    for c in range(coils):
        g.upload(c, (rng.standard_normal(N ** dim) + 1j * rng.standard_normal(N ** dim)).astype(np.complex64))
    handles = []
    for _ in range(2):
        s = hip.Samples(ctx, dim, M, coils)
        s.set_traj(t)
        handles.append(s)
    plan = hip.Plan(ctx, handles[0], N, 4.0, lut)
    out = hip.DeviceBuffer(ctx, 8 * M * coils)

    def result(call):
        out.from_host(np.zeros(2 * M * coils, np.float32))
        call()
        return out.to_host(np.int32)

    ref = result(lambda: hip.degrid_execute(plan, handles[1], g, out))
    with Capture(ctx) as graph:
        hip.degrid_execute(plan, handles[0], g, out)
    for turn in range(3):
        np.testing.assert_array_equal(result(graph.launch), ref)
        np.testing.assert_array_equal(result(lambda: hip.degrid_execute(plan, handles[0], g, out)), ref)
    graph.close()
