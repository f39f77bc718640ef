"""The device-CSR entries when the input is no index or has an id out of range: one
read-back tells, nothing is added, and the context counts on."""
import numpy as np
import pytest

import xxtric_amd

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[case]", *a, flush=True)


def _triangle(n):
    off = np.full(n + 1, 6, np.int64)
    off[:3] = 0, 2, 4
    return off, np.array([1, 2, 0, 2, 0, 1], np.int64)


@pytest.mark.parametrize("entry", ["single_gpu_count", "single_gpu_count_noalloc"])
@pytest.mark.parametrize("n", [3, 100, 5000])
def test_bad_input_adds_nothing(ctx, entry, n):
    count = ctx.to_device(np.array([40], np.int64))
    expect = 40
    for kind in ("good", "falling offsets", "late first offset", "id too large", "negative id", "unsorted", "good"):
        off, tails = _triangle(n)
        if kind == "falling offsets":
            off[1], off[2] = 4, 2
        elif kind == "late first offset":
            off[0] = 1
        elif kind == "id too large":
            tails[3] = n
        elif kind == "negative id":
            tails[0] = -1
        elif kind == "unsorted":
            tails[:2] = 2, 1
        _say(entry, n, kind)
        d_off, d_tails = ctx.to_device(off), ctx.to_device(tails)
        run = getattr(ctx, entry)
        if kind == "good":
            run(n, d_off.ptr, d_tails.ptr, count.ptr)
            expect += 1
        else:
            with pytest.raises(xxtric_amd.XtError):
                run(n, d_off.ptr, d_tails.ptr, count.ptr)
        assert int(count.download(np.int64, 1)[0]) == expect
        d_off.close()
        d_tails.close()
    count.close()
