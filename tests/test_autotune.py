"""
The autotuner's candidates and cache (no GPU): the untuned shape is timed, so that tuning never leaves a call slower
than it found it, and a winner that was cached before the untuned shape's rules changed is not taken.
"""
from __future__ import annotations

import json

import pytest
import torch

from pyocean_amd import autotune, batch


@pytest.fixture
def fake(monkeypatch, tmp_path):
    """Steps that cost what ``ms`` says; returns (calls' shapes, cache path)."""
    monkeypatch.setenv("OCX_TUNING_CACHE", str(tmp_path / "t.json"))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda d: "a GPU")
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: None)
    seen = []
    monkeypatch.setattr(batch, "set_tuning", lambda r, w: seen.append((r, w)))
    # the untuned shape is the fastest, as on a small domain whose rows the rule takes below every fixed candidate
    monkeypatch.setattr(autotune, "_time_ms", lambda fn, reps, stream: 1.0 if seen[-1] == (0, 0) else 2.0)
    return seen, tmp_path / "t.json"


def _tune(**kw):
    t = torch.zeros(1, 2, 3, 4)
    return autotune.tune_step(t, t, t, t, t, t, 1.0, **kw)


def test_the_untuned_shape_is_a_candidate_and_can_win(fake):
    seen, cache = fake
    best, table = _tune()
    assert best == autotune.Shape(0, 0) and best.tile == "untuned"
    assert seen[-1] == (0, 0)                                       # what the call leaves set
    assert [s for s, _ in table].count(best) == 1
    assert {s.rows_per_chunk for s, _ in table} >= {2, 4, 8, 64}
    assert (0, 0, 0) in autotune._candidates(autotune.BATCH_ROWS, autotune.WAVES, autotune.GROUPS)
    assert _tune() == (best, [])                                    # cached
    assert autotune._candidates((16, 64), (1, 2)) == [(16, 1), (16, 2), (64, 1), (64, 2)]
    assert autotune._candidates(iter((0, 64)), (1, 2)) == [(0, 0), (0, 1), (0, 2), (64, 1), (64, 2)]


def test_a_winner_of_older_rules_is_not_taken(fake):
    seen, cache = fake
    key = "a_GPU|step|f64|1x2x3x4"
    cache.write_text(json.dumps({key: dict(rows_per_chunk=64, waves_per_group=1, groups_per_cu=0)}))
    best, table = _tune()
    assert table and best == autotune.Shape(0, 0)
    assert autotune.cached("step", "f64", [(1, 2, 3, 4)]) == best
