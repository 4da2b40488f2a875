"""The autotuner against the library's default schedule: an entry names a candidate only
where it beats the default, whose time is the entry's default_ms; candidates and the default
are timed without the entries cached so far."""
import json

import pytest
import torch

from blockstructuredsolvers_amd import autotune, solver

A = {"chain_len_levels": [3] * 16, "base_max": 8}
B = {"chain_len_levels": [5] + [2] * 15, "base_max": 2}


@pytest.mark.parametrize("times,best", [({"default": 1.0, "A": 1.2, "B": 1.1}, {}),
                                        ({"default": 1.0, "A": 1.0, "B": 1.1}, {}),
                                        ({"default": 1.0, "A": 1.2, "B": 0.9}, B)])
def test_tune_keeps_the_default_unless_beaten(monkeypatch, tmp_path, times, best):
    def timed(cfg, *args, **kw):
        return times["default" if not cfg else "A" if cfg == A else "B"]

    monkeypatch.setattr(autotune, "_time_config", timed)
    monkeypatch.setattr(autotune, "_device_systems", lambda *a: None)
    path = str(tmp_path / "tuned.json")
    e = autotune.tune(40, 16, configs=[A, B], path=path, log=lambda m: None)
    assert e == {"config": best, "ms": min(times.values()) if best else 1.0, "default_ms": 1.0}
    assert json.load(open(path)) == {autotune.key(40, 16, torch.float64, "plain"): e}
    assert autotune.lookup(40, 16, torch.float64, "plain", path=path) == best


def test_candidates_are_timed_untuned(monkeypatch):
    class Stop(Exception):
        pass

    seen = {}

    def plan(*args, **kw):
        seen.update(kw)
        raise Stop

    monkeypatch.setattr(solver, "initialize_batched", plan)
    systems = [autotune_system()]
    with pytest.raises(Stop):
        autotune._time_config({}, systems, torch.float64, "plain", 1, None)
    assert seen["tuned"] is False


def autotune_system():
    from blockstructuredsolvers_amd import workloads
    return workloads.spd_system(4, 16)
