"""The count in rank space (totals, per-vertex counts and owned ranges, library default knobs)
at the sizes where it can go wrong: lists around one chunk, one line and
one wave, ranks on both sides of the 16-bit limit, more cold ids than one hash
holds, rows across chunks, rows of many empty neighbours, labels in any order.
Expected values: the oracle, closed forms, and the edge tiles (asked for by
setting one of their knobs)."""
import numpy as np
import pytest

import oracle_py as O
from helpers import complete, csr_from_edges, random_graph

pytestmark = pytest.mark.gpu

HOT = 65535  # ranks below are kept in 16 bits


def _say(*a):
    print("[case]", *a, flush=True)


def _tiles(ctx, g, **kw):
    ctx.tune(small_cut=32)
    try:
        return g.count(**kw)
    finally:
        ctx.tune(small_cut=-1)


def _same(a, b):
    return a[0] == b[0] and (a[1] == b[1]).all()


def _circulant(n, k):
    """Vertex i joined to i +- 1 .. k: n k (k - 1) / 2 triangles for n > 3 k."""
    step = np.concatenate([np.arange(-k, 0), np.arange(1, k + 1)])
    t = np.sort((np.arange(n, dtype=np.int64)[:, None] + step[None, :]) % n, axis=1)
    return np.arange(n + 1, dtype=np.int64) * (2 * k), t.reshape(-1)


def _beside(a, b):
    return np.concatenate([a[0], a[0][-1] + b[0][1:]]), np.concatenate([a[1], b[1] + len(a[0]) - 1])


@pytest.mark.parametrize("n", [3, 9, 10, 17, 33, 34, 65, 66, 130, 1025])
def test_list_lengths(ctx, n):
    """K_n: lists of every length up to n - 1, around chunk, line, lane and wave sizes."""
    _say("complete", n)
    off = np.arange(n + 1, dtype=np.int64) * (n - 1)
    cols = np.tile(np.arange(n, dtype=np.int64), n).reshape(n, n)
    tails = cols[~np.eye(n, dtype=bool)].reshape(-1)
    assert ctx.count_csr(off, tails) == n * (n - 1) * (n - 2) // 6
    i = np.arange(n, dtype=np.int64)
    tot, pv = ctx.count_csr(off, tails, per_vertex=True)   # from 512 ids on: beyond the slots in LDS
    assert tot == n * (n - 1) * (n - 2) // 6 and (pv == (n - 1 - i) * (n - 2 - i) // 2).all()


@pytest.mark.parametrize("n", [HOT - 1, HOT, HOT + 1, HOT + 2, HOT + 70])
def test_ranks_around_the_hot_limit(ctx, n):
    """All degrees equal, so any vertex may take the ranks on either side."""
    k = 5
    _say("circulant", n, k)
    off, tails = _circulant(n, k)
    assert ctx.count_csr(off, tails) == n * k * (k - 1) // 2
    for orient in ("degree", "id"):
        _say(orient)
        tot, pv = ctx.count_csr(off, tails, per_vertex=True, orient=orient)
        assert tot == n * k * (k - 1) // 2 == int(pv.sum())
        assert (pv[:n - 2 * k] [2 * k:] == k * (k - 1) // 2).all()  # rows that do not wrap


@pytest.mark.parametrize("k,clique", [(34, 64), (110, 200), (600, 1150)])
def test_cold_lists(ctx, k, clique):
    """65,600 vertices of degree 2k outrank a clique of smaller degree: its lists are all
    cold ids -- within the small hash, past it, and more than one filling of the large one."""
    n = 65600
    _say("circulant and clique", k, clique)
    i = np.arange(clique, dtype=np.int64)
    cols = np.tile(i, clique).reshape(clique, clique)[~np.eye(clique, dtype=bool)].reshape(-1)
    off, tails = _beside(_circulant(n, k), (np.arange(clique + 1, dtype=np.int64) * (clique - 1), cols))
    g = ctx.graph(off, tails.astype(np.int32))
    exp = n * k * (k - 1) // 2 + clique * (clique - 1) * (clique - 2) // 6
    assert g.count() == exp
    assert ctx.timing()["ne_plus"] == len(tails) // 2
    if len(tails) < 1 << 25:
        tot, pv = g.count(per_vertex=True)
        assert tot == exp and (pv[n:] == (clique - 1 - i) * (clique - 2 - i) // 2).all()
        assert int(pv.sum(dtype=np.uint64)) == exp
    g.close()


@pytest.mark.parametrize("make", ["empty_between", "self_loops", "star", "two_hubs", "isolated_tail"])
def test_row_shapes(ctx, make):
    _say(make)
    rng = np.random.default_rng(4)
    if make == "empty_between":    # every 700th vertex has edges: chunks span thousands of empty rows
        a = rng.integers(0, 300, (4000, 2)) * 700
        off, tails = csr_from_edges(300 * 700, [(int(x), int(y)) for x, y in a if x != y])
    elif make == "self_loops":
        a = rng.integers(0, 900, (9000, 2))
        off, tails = csr_from_edges(900, [(int(x), int(y)) for x, y in a] + [(i, i) for i in range(0, 900, 7)])
    elif make == "star":           # one row across dozens of chunks, closed by a path
        n = 50001
        off, tails = csr_from_edges(n, [(0, i) for i in range(1, n)] + [(i, i + 1) for i in range(1, n - 1)])
    elif make == "two_hubs":       # a row ends and the next begins inside a chunk, both longer than it
        n = 9000
        off, tails = csr_from_edges(n, [(0, 1)] + [(h, i) for h in (0, 1) for i in range(2, n)])
    else:                          # one edge, then rows without any
        off, tails = csr_from_edges(5000, [(0, 1), (1, 2), (0, 2)])
    exp = O.count_degree_ordered(off, tails.astype(np.int32))
    assert ctx.count_csr(off, tails) == exp
    g = ctx.graph(off, tails)
    assert g.count() == exp and _tiles(ctx, g) == exp
    ref = O.count_reference(off, tails.astype(np.int32), per_vertex=True)
    for orient in ("degree", "id"):
        assert _same(g.count(per_vertex=True, orient=orient), ref) and g.count(orient=orient) == exp
    g.close()


@pytest.mark.parametrize("scale,permute", [(9, True), (13, False), (17, True), (17, False), (20, True)])
def test_rmat_equals_the_edge_tiles(ctx, scale, permute):
    _say("rmat", scale, permute)
    g = ctx.rmat(scale, 16, 5, permute)
    a = g.count()
    assert a == _tiles(ctx, g) == g.count(orient="id")
    assert _same(g.count(per_vertex=True), _tiles(ctx, g, per_vertex=True))
    if scale <= 17:
        assert a == O.count_degree_ordered(*g.download())
    g.close()


@pytest.mark.parametrize("orient", ["degree", "id"])
@pytest.mark.parametrize("n", [70, 5000, 90000])
def test_host_csr_per_vertex(ctx, n, orient):
    """Short rows, also past the 16-bit limit (cold lists), against the reference restatement."""
    import xxtric_amd
    off, tails = xxtric_amd.rgg_generate(n, seed=3, connect=True, strict=True)
    _say("rgg", n, orient)
    exp = O.count_reference(off, tails.astype(np.int32), per_vertex=True)
    assert _same(ctx.count_csr(off, tails, per_vertex=True, orient=orient), exp)
    assert ctx.count_csr(off, tails, orient=orient) == exp[0]


@pytest.mark.parametrize("make", ["rgg90000", "circulant", "rmat17", "rmat13 unpermuted"])
def test_owned_ranges(ctx, make):
    """Owned ranges at the ends, in the middle, empty and whole, with cold lists: the owned
    count against the per-vertex counts, both against the edge tiles."""
    import xxtric_amd
    if make == "rgg90000":
        g = ctx.graph(*xxtric_amd.rgg_generate(90000, seed=5, connect=True, strict=True))
    elif make == "circulant":
        g = ctx.graph(*_circulant(HOT + 300, 40))
    else:
        g = ctx.rmat(int(make[4:6]), 16, 4, make == "rmat17")
    _, pv = g.count(per_vertex=True)
    n = g.nv
    for lo, hi in ((0, n // 8), (n // 3, n // 2), (n - n // 8, n), (0, n), (7, 7), (n - 1, n), (100, 164)):
        _say(make, lo, hi)
        owned, local, _ = g.count_owned(lo, hi, total=False)
        ne_plus = ctx.timing()["ne_plus"]
        assert owned == int(pv[lo:hi].sum(dtype=np.uint64))
        ctx.tune(small_cut=32)
        try:
            assert (owned, local) == g.count_owned(lo, hi, total=False)[:2]
            assert ne_plus == ctx.timing()["ne_plus"]
        finally:
            ctx.tune(small_cut=-1)
    g.close()


def test_device_csr_and_graph_sizes_in_a_row(ctx):
    """The reference launcher's int64 CSR, and scratch that is kept from larger graphs."""
    for off, tails in (O.rmat_csr(15, 16, 3, True), complete(40), random_graph(200, 0.2, 9), O.rmat_csr(12, 16, 3, False)):
        _say("device csr", len(off) - 1)
        d = [ctx.to_device(np.asarray(x, np.int64)) for x in (off, tails, [11])]
        ctx.single_gpu_count(len(off) - 1, d[0].ptr, d[1].ptr, d[2].ptr)
        assert int(d[2].download(np.int64, 1)[0]) == 11 + O.count_degree_ordered(off, np.asarray(tails, np.int32))
        for b in d:
            b.close()


def test_ids_out_of_range_are_reported(ctx):
    from xxtric_amd import XtError, capi
    off, tails = complete(30)
    tails = tails.astype(np.int32)
    tails[17] = 30
    g = ctx.graph(off, tails)
    with pytest.raises(XtError) as e:
        g.count()
    assert e.value.code == capi.XT_ERR_INPUT
    g.close()
