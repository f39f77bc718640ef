"""Input that is no index is refused before a kernel walks it, and the context counts on."""
import numpy as np
import pytest

import xxtric_amd
from xxtric_amd import capi

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[case]", *a, flush=True)


@pytest.mark.parametrize("middle", [(4, 2, 4), (2 ** 62, -2 ** 63, -2 ** 62), (3, -2 ** 63, 4), (2 ** 63 - 1, -2, 4)])
def test_host_offsets_that_step_down(ctx, middle):
    """Also where the step does not fit 64 bits, so that the difference looks like a step up."""
    off = np.array((0,) + middle + (6,), np.int64)
    tails = np.array([1, 2, 0, 2, 0, 1], np.int64)
    _say(off.tolist())
    for call in (lambda: ctx.count_csr(off, tails), lambda: ctx.graph(off, tails)):
        with pytest.raises(xxtric_amd.XtError) as e:
            call()
        assert e.value.code == capi.XT_ERR_INPUT
    assert ctx.count_csr(np.array([0, 2, 4, 6, 6], np.int64), tails) == 1


@pytest.mark.parametrize("entry", ["single_gpu_count", "single_gpu_count_noalloc"])
@pytest.mark.parametrize("last", [6, 2 ** 31 + 5, 2 ** 42, 2 ** 43 + 7, 2 ** 45, 2 ** 62])
def test_device_offsets_that_step_down(ctx, entry, last):
    """The number of entries is read from a device array that may be no index: whatever
    stands there, the call says so (the allocation-free entry may name its capacity)."""
    off, tails = np.array([0, 4, 2, last], np.int64), np.array([1, 2, 0, 2, 0, 1], np.int64)
    _say(entry, off.tolist())
    d = [ctx.to_device(x) for x in (off, tails, np.array([5], np.int64))]
    with pytest.raises(xxtric_amd.XtError) as e:
        getattr(ctx, entry)(3, d[0].ptr, d[1].ptr, d[2].ptr)
    assert e.value.code == capi.XT_ERR_INPUT or (entry.endswith("noalloc") and e.value.code == capi.XT_ERR_CAPACITY)
    assert int(d[2].download(np.int64, 1)[0]) == 5
    for b in d:
        b.close()
    assert ctx.count_csr(np.array([0, 2, 4, 6], np.int64), tails) == 1
