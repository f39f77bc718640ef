"""A cached choice of knobs is applied only where its search started from the defaults
of today: one made among edge tiles alone says nothing about rank space."""
import json

import pytest

from xxtric_amd import autotune


class _Context:
    def __init__(self):
        self.calls = []

    def tune(self, **kw):
        self.calls.append(kw)


BEST = {"light_cut": 32, "wave_owner": 128, "group_round": 2, "group_blocks": 4, "items_per_tile": 256,
        "tile_run": 16, "group_hash": 2, "ms": 340.1}


@pytest.mark.parametrize("start,applied", [
    (None, False),  # as written before there was a choice besides the edge tiles
    ({"light_cut": 32, "wave_owner": 256, "group_round": 2, "group_blocks": 4, "items_per_tile": 256, "tile_run": 16,
      "group_hash": 1}, False),
    (autotune.DEFAULTS, True)])
def test_choice_of_another_default_is_left(tmp_path, start, applied):
    cache = str(tmp_path / "tuning.json")
    entry = {"best": BEST, "default_ms": 350.0, "trials": []}
    if start is not None:
        entry["start"] = start
    with open(cache, "w") as f:
        json.dump({"rmat_s26": entry}, f)
    c = _Context()
    got = autotune.apply_cached(c, "rmat_s26", cache=cache)
    assert (got is not None) == applied and len(c.calls) == (1 if applied else 0)
    if applied:
        assert got["wave_owner"] == 128 and c.calls[0]["small_cut"] == 32
    assert autotune.apply_cached(c, "rmat_s22", cache=cache) is None
