"""The autotuner's choices on timings that are given (no device calls: runs without a
GPU): the built-in rule is among the candidates and is kept where nothing is faster."""
import types

import numpy as np
import pytest

from channel import tuning


@pytest.fixture
def tuned(monkeypatch):
    """Replaces the library; seconds(shapes) stands for a window's time."""
    def run(seconds, members=4):
        shapes = {}
        fake = types.SimpleNamespace(
            sc_set_tuning=shapes.__setitem__, sc_set_members=lambda n: None,
            sc_set_precision=lambda m: None, c_init=lambda *a: 0, c_destroy=lambda: None)
        monkeypatch.setattr(tuning, "c_channel", fake)
        monkeypatch.setattr(tuning, "_window", lambda states, steps: seconds(shapes))
        best = tuning.autotune((16, 33, 12), (1.0, 1.0), 2000.0, 4.0 / 3.0, 0.01,
                               np.zeros((members, 12, 2, 31, 8), complex))
        assert shapes == best
        return best
    return run


def test_rule_kept_where_nothing_is_faster(tuned):
    best = tuned(lambda s: 1.0 + sum(0.1 for v in s.values() if v))
    assert best == {name: 0 for name in tuning.SHAPES}


def test_faster_shape_chosen(tuned):
    best = tuned(lambda s: 1.0 - 0.1 * (s["rebuild_blocks"] == 64) + 0.1 * (s["force_blocks"] > 0))
    assert best["rebuild_blocks"] == 64 and best["force_blocks"] == 0
