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
