"""Batches of graphs of up to 65,535 vertices (16-bit lists), and the line to larger
ones: rows around a lane's registers, a step and a sweep of list chunks, rows across
chunks, self-loops, graphs around the 16-bit limit behind other graphs, many tiny
graphs.  Expected values: the oracle and closed forms."""
import numpy as np
import pytest

import oracle_py as O
import xxtric_amd
from helpers import complete, csr_from_edges, random_graph
from xxtric_amd import XT_BATCH_HIPGRAPH, XT_BATCH_PERSISTENT

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[case]", *a, flush=True)


def _run(ctx, graphs, exp):
    b = xxtric_amd.Batch(ctx, sum(len(o) - 1 for o, _ in graphs), max(1, sum(len(t) for _, t in graphs)), len(graphs))
    for off, tails in graphs:
        b.add(off, tails)
    for orient in ("degree", "id"):
        for mode in (XT_BATCH_PERSISTENT, XT_BATCH_HIPGRAPH, XT_BATCH_HIPGRAPH):
            _say(orient, mode)
            b.run(mode, orient)
            assert [int(x) for x in b.results()] == [int(x) for x in exp]
    b.close()


def _circulant(n, k):
    """Vertex i joined to i +- 1 .. k: n k (k - 1) / 2 triangles for n > 3 k."""
    step = np.concatenate([np.arange(-k, 0), np.arange(1, k + 1)])
    t = np.sort((np.arange(n, dtype=np.int64)[:, None] + step[None, :]) % n, axis=1)
    return np.arange(n + 1, dtype=np.int64) * (2 * k), t.reshape(-1)


@pytest.mark.parametrize("sizes", [(1, 2, 3), (9, 10, 11), (17, 18, 65, 66, 67), (513, 3, 514), (600, 600), (1100,)])
def test_list_lengths(ctx, sizes):
    """K_n: lists of every length up to n - 1, so rows around 8, 64 and 512 ids."""
    _say("complete", sizes)
    _run(ctx, [complete(n) for n in sizes], [n * (n - 1) * (n - 2) // 6 for n in sizes])


@pytest.mark.parametrize("n", [65534, 65535, 65536])
def test_vertices_around_the_limit(ctx, n):
    """The last takes the batch to the edge tiles; the graphs before it move its ids."""
    _say("circulant", n)
    small = [complete(5), random_graph(300, 0.1, 3)]
    exp = [O.count_degree_ordered(*g) for g in small]
    for k in (3, 12):
        _run(ctx, small + [_circulant(n, k), small[1]], exp + [n * k * (k - 1) // 2, exp[1]])


@pytest.mark.parametrize("seed", [1, 2])
def test_shapes(ctx, seed):
    """Hubs and empty rows, self-loops, graphs of a few vertices between large ones."""
    rng = np.random.default_rng(seed)
    graphs = []
    for i in range(60):
        n = int(rng.integers(1, 12)) if i % 3 else int(rng.integers(50, 3000))
        m = int(rng.integers(0, 12 * n))
        u = (n * rng.random(m) ** 3).astype(np.int64)
        v = rng.integers(0, n, m)
        graphs.append(csr_from_edges(n, list(zip(u.tolist(), v.tolist()))))
    n = 4000  # one vertex joined to all: a row of many chunks
    graphs.append(csr_from_edges(n, [(0, i) for i in range(1, n)] +
                                 list(zip(rng.integers(1, n, 9000).tolist(), rng.integers(1, n, 9000).tolist()))))
    _say("shapes", seed, len(graphs))
    _run(ctx, graphs, [O.count_degree_ordered(*g) for g in graphs])
