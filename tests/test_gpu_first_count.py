"""The reported device times of a context's first count hold the kernels alone: the
scratch that it allocates is not in them."""
import time

import pytest

import xxtric_amd

pytestmark = pytest.mark.gpu


def test_allocations_are_not_timed(ctx):
    g = ctx.rmat(18, 16, 1, True)
    g.count()  # the kernels are loaded
    g.close()
    allocs = inside = 0.0
    for _ in range(3):
        with xxtric_amd.Context(0) as c:
            g = c.rmat(18, 16, 1, True)
            wall, dev = [], []
            for _ in range(4):
                t = time.perf_counter()
                g.count()
                wall.append((time.perf_counter() - t) * 1e3)
                dev.append(c.timing()["total_ms"])
            g.close()
        # What the first call takes longer than a later one is its allocations.
        allocs += wall[0] - min(wall[1:])
        inside += dev[0] - min(dev[1:])
        print("[case] first calls longer by %.3f ms, their device times by %.3f ms" % (allocs, inside), flush=True)
    assert allocs > 0 and inside < 0.5 * allocs
