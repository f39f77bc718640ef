"""Per-vertex counts in rank space around the places a wave has slots for, and with
steps of few and of many hits, credited to each of a triangle's three vertices
(labels ascending, descending and shuffled against the ranks).  Expected: closed
forms and the edge tiles (asked for by setting one of their knobs)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[case]", *a, flush=True)


def _tiles(ctx, g, **kw):
    ctx.tune(small_cut=32)
    try:
        return g.count(**kw)
    finally:
        ctx.tune(small_cut=-1)


@pytest.mark.parametrize("n", [64, 129, 1023, 1024, 1025, 1026, 1500])
def test_places_around_the_slots(ctx, n):
    _say("complete", n)
    off = np.arange(n + 1, dtype=np.int64) * (n - 1)
    cols = np.tile(np.arange(n, dtype=np.int64), n).reshape(n, n)
    tot, pv = ctx.count_csr(off, cols[~np.eye(n, dtype=bool)].reshape(-1), per_vertex=True)
    i = np.arange(n, dtype=np.int64)
    assert tot == n * (n - 1) * (n - 2) // 6 and (pv == (n - 1 - i) * (n - 2 - i) // 2).all()


@pytest.mark.parametrize("labels", ["by degree", "against degree", "shuffled"])
@pytest.mark.parametrize("n,power", [(700, 0.0), (3000, 1.0), (9000, 2.0)])
def test_credit_by_label(ctx, n, power, labels):
    """Edges with a skew by vertex; a dense graph (every id of a chunk hits) without one."""
    rng = np.random.default_rng(n)
    m = 200_000
    u, v = (np.minimum((n * rng.random(m) ** (1 + power)).astype(np.int64), n - 1) for _ in range(2))
    name = np.arange(n) if labels == "by degree" else np.arange(n)[::-1] if labels == "against degree" else rng.permutation(n)
    g = ctx.graph_from_edges(n, name[u], name[v])
    _say(n, power, labels)
    a, b = g.count(per_vertex=True), _tiles(ctx, g, per_vertex=True)
    g.close()
    assert a[0] == b[0] and (a[1] == b[1]).all()


@pytest.mark.parametrize("d", [63, 64, 65, 128, 255, 256, 257, 320, 512, 600])
def test_rows_around_a_block_of_loads(ctx, d):
    """Two rows of d smaller ranks (and one more) under d mutually joined hubs that a
    fringe of pendant vertices lifts above them."""
    rng = np.random.default_rng(d)
    hubs = np.arange(d, dtype=np.int64)
    a, b = np.triu_indices(d, 1)
    u = [hubs[a], np.repeat([d, d + 1], d), np.array([d])]
    v = [hubs[b], np.tile(hubs, 2), np.array([d + 1])]
    n = d + 2 + 4 * d
    u.append(np.repeat(hubs, 4))
    v.append(np.arange(d + 2, n))
    name = rng.permutation(n)
    g = ctx.graph_from_edges(n, name[np.concatenate(u)], name[np.concatenate(v)])
    _say("hubs", d)
    total = d * (d - 1) * (d - 2) // 6 + 2 * (d * (d - 1) // 2) + d
    assert g.count() == total
    a, b = g.count(per_vertex=True), _tiles(ctx, g, per_vertex=True)
    g.close()
    assert a[0] == b[0] == total and (a[1] == b[1]).all()
