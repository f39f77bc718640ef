"""A context with library defaults counts in rank space (own contexts here, so that no
knob another test has set can hide it), and rows of many cold ids (ranks from 65,535
on), which take several fillings of the hash, are credited right per vertex and to an
owned range.  Expected values: closed forms."""
import numpy as np
import pytest

import xxtric_amd

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[case]", *a, flush=True)


@pytest.fixture(scope="module")
def own():
    with xxtric_amd.Context(0) as c:
        yield c


def _ranked(c):
    t = c.timing()  # rank space has no item lists, and every edge is its group phase's
    return t["items_ms"] == 0 and t["n_heavy"] == t["ne_plus"] > 0 and t["group_ms"] > 0


def test_defaults_count_in_rank_space(own):
    off, tails = xxtric_amd.rgg_generate(5000, seed=3)
    n = len(off) - 1
    total = own.count_csr(off, tails)
    assert _ranked(own)
    own.tune(small_cut=32)
    assert own.count_csr(off, tails) == total and not _ranked(own)
    own.tune(small_cut=-1)
    for orient in ("degree", "id"):
        assert own.count_csr(off, tails, per_vertex=True, orient=orient)[0] == total and _ranked(own), orient
    for make in (lambda: own.graph(off, tails), lambda: own.rmat(12, 16, 1, True)):
        g = make()
        _say("resident", g.nv)
        g.count()
        assert _ranked(own)
        g.count(per_vertex=True)
        assert _ranked(own)
        g.count_owned(0, g.nv // 2, total=False)
        assert _ranked(own)
        g.close()
    u = np.repeat(np.arange(n), np.diff(off))
    assert own.count_edges(n, u, tails) == total and _ranked(own)


@pytest.mark.parametrize("k,clique", [(110, 200), (600, 1150)])
def test_cold_rows(own, k, clique):
    """65,600 vertices of degree 2k outrank a clique of smaller degree; as many vertices
    without edges follow as keep the graph from counting as dense."""
    n = 65600
    step = np.concatenate([np.arange(-k, 0), np.arange(1, k + 1)])
    ring = np.sort((np.arange(n, dtype=np.int64)[:, None] + step[None, :]) % n, axis=1).astype(np.int32).reshape(-1)
    i = np.arange(clique, dtype=np.int64)
    cols = np.tile(i, clique).reshape(clique, clique)[~np.eye(clique, dtype=bool)].reshape(-1)
    off = np.concatenate([np.arange(n, dtype=np.int64) * 2 * k, n * 2 * k + np.arange(clique + 1, dtype=np.int64) * (clique - 1)])
    off = np.concatenate([off, np.full(int(off[-1]) // 64, off[-1])])
    g = own.graph(off, np.concatenate([ring, (cols + n).astype(np.int32)]))
    _say("circulant and clique", k, clique)
    in_ring, in_clique = n * k * (k - 1) // 2, clique * (clique - 1) * (clique - 2) // 6
    credit = (clique - 1 - i) * (clique - 2 - i) // 2  # of clique vertex i: pairs of larger ones
    tot, pv = g.count(per_vertex=True)
    assert _ranked(own)
    assert tot == in_ring + in_clique == int(pv.sum(dtype=np.uint64)) and (pv[n:n + clique] == credit).all()
    for lo, hi in ((0, clique), (0, 1), (clique // 10, clique // 2), (clique // 2, clique)):
        _say("owned", lo, hi)
        owned, local, _ = g.count_owned(n + lo, n + hi, total=False)
        assert _ranked(own)
        # Smallest vertex a and middle vertex b owned: b's larger neighbours, for each a below b.
        middle = i[lo:hi]
        assert owned == int(credit[lo:hi].sum()) and local == int(((middle - lo) * (clique - 1 - middle)).sum())
    assert g.count_owned(0, n, total=False)[0] == in_ring
    g.close()
