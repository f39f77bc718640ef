"""Graphs of an odd shape, where counting in rank space once took several times as long
as with edge tiles (asked for by setting one of their knobs): not slower than half
again now."""
import numpy as np
import pytest

import xxtric_amd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def own():
    with xxtric_amd.Context(0) as c:
        yield c


def _ms(c, call):
    call()
    out = []
    for _ in range(5):
        result = call()
        out.append(c.timing()["total_ms"])
    return float(np.median(out)), result


def _against_tiles(c, g, **kw):
    a, ra = _ms(c, lambda: g.count(**kw))
    c.tune(small_cut=32)
    b, rb = _ms(c, lambda: g.count(**kw))
    c.tune(small_cut=-1)
    g.close()
    print("[case]", kw, "%.3f ms, edge tiles %.3f ms" % (a, b), flush=True)
    if kw.get("per_vertex"):
        assert ra[0] == rb[0] and (ra[1] == rb[1]).all()
    else:
        assert ra == rb
    assert a <= 1.5 * b


def test_a_hub_of_thousands_of_chunks(own):
    """The chunks that a row of 2,000,000 entries bounds are marked by a wave, not a lane."""
    n = 2_000_000
    u = np.concatenate([np.zeros(n - 1, np.int64), np.arange(1, n - 1)])
    v = np.concatenate([np.arange(1, n), np.arange(2, n)])
    _against_tiles(own, own.graph_from_edges(n, u, v))


@pytest.mark.parametrize("clique,copies", [(1000, 1), (2000, 1), (200, 800), (1200, 12)])
def test_per_vertex_counts_of_dense_graphs(own, clique, copies):
    """Where nearly every id that is looked up is a hit, and out-lists are long."""
    a, b = np.triu_indices(clique, 1)
    base = (np.arange(copies) * clique)[:, None]
    _against_tiles(own, own.graph_from_edges(clique * copies, (base + a).reshape(-1), (base + b).reshape(-1)), per_vertex=True)
