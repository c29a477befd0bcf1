"""Device memory that a context keeps from closed plans."""
import ctypes as C
import time

import numpy as np
import pytest

from fastrecon_amd import hip

pytestmark = pytest.mark.gpu


def free_bytes():
    """Free device memory, once it no longer changes (the driver frees in the background)."""
    last = [-1, -2]
    while len(set(last[-4:])) > 1:
        time.sleep(0.1)
        last.append(reported())
    return last[-1]


def reported():
    runtime = C.CDLL("libamdhip64.so")               # the copy the library has loaded
    free, total = C.c_size_t(), C.c_size_t()
    assert runtime.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_trim():
    ctx = hip.Context(0)
    rng = np.random.default_rng(0)
    M, N = 2_000_000, 96
    s = hip.Samples(ctx, 3, M, 1)
    s.set_traj(rng.uniform(0, N - 1, (M, 3)).astype(np.float32))
    lut, _ = hip.kb_lut(4.0, 2.0, 512)
    hip.Plan(ctx, s, N, 4.0, lut).close()            # what the runtime takes for the first launches
    ctx.trim()
    before = free_bytes()
    hip.Plan(ctx, s, N, 4.0, lut).close()
    kept = before - free_bytes()
    ctx.trim()
    left = before - free_bytes()
    print(f"[pool] {kept >> 20} MiB kept, {left >> 20} MiB after the trim", flush=True)
    assert kept >= 200 << 20                         # a build sorts 16M records, 16 bytes each
    assert left <= 16 << 20                          # (small blocks share pages)
    hip.Plan(ctx, s, N, 4.0, lut).close()            # and it serves again
    s.close()
    ctx.close()
