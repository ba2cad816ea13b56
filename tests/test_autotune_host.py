"""The tuner's choice and its cache, without a GPU (no counterpart in the reference)."""
import json
import math

import numpy as np
import pytest

from halotools_amd import autotune


@pytest.fixture
def cache(tmp_path, monkeypatch):
    monkeypatch.setenv("HALOTOOLS_AMD_TUNE_CACHE", str(tmp_path / "tune.json"))
    monkeypatch.setattr(autotune, "_CACHE", {})
    return tmp_path / "tune.json"


def test_the_librarys_own_choice_is_timed_and_stays_unless_clearly_slower():
    own = (0.0, 0)
    assert 0.0 in autotune.TARGETS and {0, 1} <= set(autotune.WAVES)
    assert autotune.cell_edge(0.0, 10 ** 6, [1000.0] * 3, 50.0) == 0.0
    assert autotune._pick({own: 1.01, (8.0, 4): 1.0}) == own
    assert autotune._pick({own: 1.10, (8.0, 4): 1.0, (8.0, 8): 1.2}) == (8.0, 4)
    assert autotune._pick({(2.0, 2): 1.0, (8.0, 8): 0.9}) == (8.0, 8)


def test_entries_of_other_kernels_are_not_found(cache):
    n, period, rmax = 100000, [500.0] * 3, 25.0
    dens = int(round(math.log2(n / float(np.prod(period)))))
    old = "%d:%d:%d" % (1, dens, int(round(4 * math.log2(rmax / 500.0))))
    cache.write_text(json.dumps({old: {"target": 8.0, "waves": 2}}))
    assert autotune.lookup(1, n, period, rmax) is None
    autotune._CACHE[autotune.key(1, n, period, rmax)] = {"target": 0.0, "waves": 1}
    autotune._save()
    assert autotune.lookup(1, n, period, rmax) == (0.0, 1)
