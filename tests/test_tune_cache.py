"""The tuner's cache and defaults, on the CPU: choices timed on other kernels
are timed again, and without timing the first candidate is taken."""
import json
import types

import pytest
import torch

import tensormesh_amd as tm
from tensormesh_amd import tune
from tensormesh_amd.mesh import unit_square_tri

DEV = torch.device("cpu")


@pytest.fixture
def clock(monkeypatch):
    """Device events that read a counter which the candidates advance."""
    now = types.SimpleNamespace(t=0.0)

    class Event:
        def __init__(self, enable_timing=True):
            pass

        def record(self):
            self.t = now.t

        def elapsed_time(self, other):
            return other.t - self.t
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    return now


def _candidates(clock, **cost):
    def run(name):
        clock.t += cost[name]
    return {n: (lambda n=n: run(n)) for n in cost}


def test_choices_of_other_kernels_are_timed_again(clock, tmp_path):
    path = tmp_path / "tune.json"
    path.write_text(json.dumps({"key": {"choice": "slow", "ms": {}}}))   # no revision: timed before there was one
    t = tune.Tuner(path)
    assert t.choose("key", _candidates(clock, slow=3.0, fast=1.0), device=DEV) == "fast"
    stored = json.loads(path.read_text())
    (key,) = [k for k in stored if k != "key"]
    assert key.startswith("key") and str(tune.KERNELS) in key
    stored[key]["choice"] = "slow"                                       # this revision's choice stays
    path.write_text(json.dumps(stored))
    assert tune.Tuner(path).choose("key", _candidates(clock, slow=3.0, fast=1.0), device=DEV) == "slow"


def test_the_kernels_own_count_is_a_candidate(clock, tmp_path, monkeypatch):
    m = unit_square_tri(2)
    A = tm.LinearElasticityElementAssembler.from_mesh(m, E=1.0, nu=0.3)
    A.epw = "auto"
    cost = {0: 1.0, 1: 3.0, 2: 2.0}
    seen = []

    def run(e):
        seen.append(e)
        clock.t += cost[e]
        return A.epw
    monkeypatch.setattr(tune, "_TUNER", tune.Tuner(tmp_path / "tune.json"))
    assert A._launch_epw("wave", DEV, torch.float64, "form", run, (1, 2)) == 0
    assert set(seen) == {0, 1, 2} and A.epw == "auto"
    monkeypatch.setenv("TENSORMESH_AMD_TUNE", "0")
    monkeypatch.setattr(tune, "_TUNER", None)
    assert A._launch_epw("wave", DEV, torch.float64, "other", run, (1, 2)) == 0
