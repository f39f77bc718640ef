"""Counts in rank space whose lists find no room (the list memory cut short) are made
with edge tiles: every entry point gives the same counts as with all its room.
Expected values: the reference restatement."""
import numpy as np
import pytest

import oracle_py as O
import xxtric_amd

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[case]", *a, flush=True)


@pytest.fixture(scope="module")
def own():
    with xxtric_amd.Context(0) as c:  # library defaults, whatever other tests set
        yield c


@pytest.mark.parametrize("lines", [16, 1024, 0])
@pytest.mark.parametrize("make", ["rmat13", "rgg20000"])
def test_short_list_memory(own, make, lines):
    off, tails = O.rmat_csr(13, 16, 5, True) if make == "rmat13" else xxtric_amd.rgg_generate(20000, seed=3)
    off, tails = np.asarray(off, np.int64), np.asarray(tails, np.int64)
    n = len(off) - 1
    total, pv = O.count_reference(off, tails.astype(np.int32), per_vertex=True)
    _say(make, lines)
    own.limit_lists(lines)
    try:
        def tiles():  # rank space has no item lists
            return own.timing()["items_ms"] > 0
        assert own.count_csr(off, tails) == total and tiles() == (lines > 0)
        for orient in ("degree", "id"):
            t, p = own.count_csr(off, tails, per_vertex=True, orient=orient)
            assert t == total and (p == pv).all()
        g = own.graph(off, tails)
        assert g.count() == total and tiles() == (lines > 0)
        for lo, hi in ((0, n // 8), (n // 3, n)):
            owned, _, t = g.count_owned(lo, hi)
            assert owned == int(pv[lo:hi].sum(dtype=np.uint64)) and t == total
        g.close()
        d = [own.to_device(x) for x in (off, tails, np.array([7], np.int64))]
        own.single_gpu_count(n, d[0].ptr, d[1].ptr, d[2].ptr)
        assert int(d[2].download(np.int64, 1)[0]) == 7 + total
        for b in d:
            b.close()
    finally:
        own.limit_lists(0)
