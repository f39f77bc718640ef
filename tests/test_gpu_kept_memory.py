"""Device memory that a context keeps (of graph builds, and of the way to count that
the running call does not take) is given back when an allocation fails, and memory that
is in use is not.  Failures are injected; every count is checked."""
import numpy as np
import pytest

import oracle_py as O
import xxtric_amd
from xxtric_amd import capi

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[case]", *a, flush=True)


def _nomem(call):
    with pytest.raises(xxtric_amd.XtError) as e:
        call()
    assert e.value.code == capi.XT_ERR_NOMEM


def _pairs(off, tails):
    u = np.repeat(np.arange(len(off) - 1), np.diff(off))
    return u, np.asarray(tails, np.int64)


@pytest.fixture(scope="module")
def graphs():
    out = {}
    for s in (10, 13):
        off, tails = O.rmat_csr(s, 16, 5, True)
        out[s] = np.asarray(off, np.int64), np.asarray(tails, np.int64), O.count_degree_ordered(off, np.asarray(tails, np.int32))
    return out


def test_build_memory_is_given_back(graphs):
    off, tails, exp = graphs[13]
    with xxtric_amd.Context(0) as c:
        _say("nothing to give")
        c.fail_tries(1)
        _nomem(lambda: c.count_csr(off, tails))
    with xxtric_amd.Context(0) as c:
        g = c.graph_from_edges(len(off) - 1, *_pairs(off, tails))  # the context keeps the build's memory
        _say("build memory for a count")
        c.fail_tries(1)
        assert g.count() == exp
        g.close()


def test_scratch_of_the_other_way_to_count(graphs):
    off, tails, exp = graphs[13]
    with xxtric_amd.Context(0) as c:
        assert c.count_csr(off, tails) == exp
        _say("rank space's scratch for edge tiles")
        c.tune(small_cut=32)
        c.fail_tries(1)
        assert c.count_csr(off, tails) == exp and c.timing()["items_ms"] > 0
        _say("edge tiles' scratch for rank space")
        c.tune(small_cut=-1)
        c.fail_tries(1)
        assert c.count_csr(off, tails) == exp and c.timing()["items_ms"] == 0
        c.tune(small_cut=32)
        assert c.count_csr(off, tails) == exp
        _say("for a graph")
        c.tune(small_cut=-1)
        assert c.count_csr(off, tails) == exp
        c.fail_tries(1)
        g = c.graph(off, tails)
        assert g.count() == exp
        g.close()


def test_memory_in_use_stays(graphs):
    """The CSR of an edge list lies in the build's memory while it is counted."""
    with xxtric_amd.Context(0) as c:
        off, tails, exp = graphs[13]
        g = c.graph_from_edges(len(off) - 1, *_pairs(off, tails))
        g.close()
        off, tails, exp = graphs[10]  # fits the memory of the larger build with its CSR
        _say("edge list")
        c.fail_tries(1)
        _nomem(lambda: c.count_edges(len(off) - 1, *_pairs(off, tails)))
        for _ in range(2):
            assert c.count_edges(len(off) - 1, *_pairs(off, tails)) == exp
        c.fail_tries(1)  # lent no longer: a batch gets it
        b = xxtric_amd.Batch(c, 1 << 12, 1 << 18, 4)
        b.add(off, tails.astype(np.int32))
        b.run()
        assert int(b.results()[0]) == exp
        b.close()
