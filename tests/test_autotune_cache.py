"""Saved launch tunings: applied without trials, unless they were saved when the parameters meant
something else (no GPU: the library's call is replaced)."""

import json

import pytest

from helpers import load_pkg


@pytest.mark.parametrize("rule,trials", [(None, 1), (1, 1), ("now", 0)])
def test_saved_tunings_of_another_meaning_are_tuned_again(tmp_path, monkeypatch, rule, trials):
    pkg = load_pkg()
    cache = tmp_path / "tuning.json"
    names = ("mode", "threshold", "workgroups", "pool_slots", "trace_workgroups", "graph_iterations")
    saved = dict(zip(names, (1, 16, 2048, 1 << 21, 0, 8)))
    if rule is not None:
        saved["rule"] = pkg.TUNING_RULE if rule == "now" else rule
    cache.write_text(json.dumps({"disk": saved, "other": dict(saved)}))
    applied, calls = [], []

    class Library:
        @staticmethod
        def skg_autotune(handle, first, packets, engines, best, rate):
            calls.append(1)
            for q, v in enumerate((1, 32, 1024, 1 << 21, 0, 8)):
                best[q] = v
            return 0

    e = pkg.Engine.__new__(pkg.Engine)
    e._h = None
    monkeypatch.setattr(pkg, "lib", lambda: Library)
    monkeypatch.setattr(pkg.Engine, "tune", lambda self, *a: applied.append(a))
    monkeypatch.setattr(pkg.Engine, "tune_pipeline", lambda self, *a: applied.append(a))
    cfg, _ = e.autotune(0, cache=str(cache), key="disk")
    assert len(calls) == trials
    assert cfg["threshold"] == (32 if trials else 16)
    assert applied == ([] if trials else [(2048, 256, 16), (1, 1 << 21, 0, 8)])
    data = json.loads(cache.read_text())
    assert data["disk"]["threshold"] == cfg["threshold"] and data["disk"]["rule"] == pkg.TUNING_RULE
    assert "other" in data
    calls.clear()
    assert e.autotune(0, cache=str(cache), key="disk")[0] == cfg and not calls
