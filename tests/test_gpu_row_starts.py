"""Row starts of a CSR built on the device: long gaps of rows without entries at the
front, between and behind, a power of two of vertices (the key of dropped entries is
then below that of a row past the last), nothing but dropped entries, rows around a
block.  Expected: numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[case]", *a, flush=True)


@pytest.mark.parametrize("nv", [1, 2, 255, 256, 257, 512, 65536, 65537, 1 << 20])
@pytest.mark.parametrize("where", ["front", "back", "both ends", "middle", "loops", "none"])
def test_row_starts(ctx, nv, where):
    rng = np.random.default_rng(nv)
    m = 500
    u, v = (rng.integers(0, min(nv, 200), m) for _ in range(2))
    if where == "back":
        u, v = nv - 1 - u, nv - 1 - v
    elif where == "both ends":
        v = nv - 1 - v
    elif where == "middle":
        u, v = (x + max(0, nv // 2 - 100) for x in (u, v))
    elif where == "loops":
        v = u
    elif where == "none":
        u = v = u[:0]
    u, v = (np.clip(x, 0, nv - 1).astype(np.int64) for x in (u, v))
    _say(nv, where)
    g = ctx.graph_from_edges(nv, u, v)
    off, tails = g.download()
    g.close()
    keep = u != v
    a, b = np.concatenate([u[keep], v[keep]]), np.concatenate([v[keep], u[keep]])
    keys = np.unique(a * nv + b)
    assert (tails.astype(np.int64) == keys % nv).all() and len(tails) == len(keys)
    assert (np.asarray(off) == np.searchsorted(keys, np.arange(nv + 1, dtype=np.int64) * nv)).all()


def test_builds_share_memory(ctx):
    """Counts of edge lists on both sides of the memory that a context keeps for
    builds, between graphs that outlive them."""
    rng = np.random.default_rng(4)
    kept = []
    for nv, m in ((1000, 6000), (50, 0), (300_000, 900_000), (1000, 5000), (1 << 20, 9_000_000), (70_000, 400_000)):
        u, v = rng.integers(0, nv, (2, m))
        _say(nv, m)
        total = ctx.count_edges(nv, u, v)
        g = ctx.graph_from_edges(nv, u, v)
        assert g.count() == total
        kept.append((g, total))
    for g, total in kept:
        assert g.count() == total
        g.close()
