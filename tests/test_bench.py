"""bench.py where the reference build is absent (CPU only)."""
import json

import bench
import oracle


def test_cpu_legs_say_why_they_are_skipped(monkeypatch):
    """The per-config reference timing is left out with its reason, so that the
    line with what was measured is still printed."""
    monkeypatch.setattr(oracle, "ref_available", lambda: False)
    out = bench.cpu_configs(1)
    assert set(out) == {"skipped"} and "reference build absent" in json.dumps(out)
