"""The autotuner on the CPU, with a stand-in for the engine whose time for a
setting is known: it starts from the engine's defaults, gives the automatic
settings back where nothing is faster, and does not reuse what another build
measured."""
import types

import numpy as np
import pytest

omc = pytest.importorskip("ompmc_amd")
P = omc.phantoms

from ompmc_amd import tune  # noqa: E402

KNOBS = ("event_target", "electron_budget", "electron_turns", "streams")


class Engine:
    """run_dij takes cost(knobs) seconds of its clock; automatic knobs are 0."""

    def __init__(self, cost):
        self.cost, self.now, self.runs = cost, 0.0, []

    def run_dij(self, phantom, spectrum, bix, nbatch=10, precision=omc.FP32, form=omc.FORM_EVENT, nsplit=1, **kw):
        k = tuple(kw.get(n, 0) for n in KNOBS)
        self.runs.append(k)
        self.now += self.cost(*k)
        return None, None, None, types.SimpleNamespace(histories=1e6)


def _tune(engine, tmp_path, monkeypatch, **kw):
    monkeypatch.setattr(tune, "CACHE", str(tmp_path / "tune.json"))
    monkeypatch.setattr(tune, "time", types.SimpleNamespace(perf_counter=lambda: engine.now))
    bix = P.beamlets(nbeams=2, radius=1.0, hist_median=100, hist_range=(50, 200))
    return tune.tune_dij(engine, types.SimpleNamespace(nreg=1001), None, bix, **kw)


def test_automatic_settings_where_nothing_is_faster(tmp_path, monkeypatch):
    e = Engine(lambda t, b, u, s: 1.0 if (t, b, u, s) == (0, 0, 0, 0) else 1.01)
    best = _tune(e, tmp_path, monkeypatch)
    assert [best[n] for n in KNOBS] == [0, 0, 0, 0]


@pytest.mark.parametrize("nsplit", [1, 20])
def test_search_starts_at_the_engine_defaults(tmp_path, monkeypatch, nsplit):
    d = omc.event_defaults(nsplit=nsplit)
    e = Engine(lambda t, b, u, s: 1.0 - (0.3 if b == 3 else 0.0) - (0.1 if s == 2 else 0.0))
    best = _tune(e, tmp_path, monkeypatch, nsplit=nsplit)
    first = next(k for k in e.runs if any(k))
    assert first == (d["event_target"], d["electron_budget"], d["electron_turns"], d["streams"])
    assert best["electron_budget"] == 3 and best["streams"] == 2        # one rung from the defaults
    assert best["event_target"] == d["event_target"] and best["electron_turns"] == d["electron_turns"]
    assert best["nsplit"] == nsplit


def test_another_build_is_timed_again(tmp_path, monkeypatch):
    e = Engine(lambda t, b, u, s: 0.5 if b == 8 else 1.0)
    kw = dict(budgets=(4, 8), turns=(30,), streams=(1,), targets=(1048576,))
    assert _tune(e, tmp_path, monkeypatch, **kw)["electron_budget"] == 8
    n = len(e.runs)
    assert _tune(e, tmp_path, monkeypatch, **kw)["electron_budget"] == 8 and len(e.runs) == n     # from the cache
    other = tmp_path / "libompmc.so"
    other.write_bytes(b"another build")
    monkeypatch.setattr(tune, "LIB_PATH", str(other), raising=False)
    e.cost = lambda t, b, u, s: 0.5 if b == 4 else 1.0
    assert _tune(e, tmp_path, monkeypatch, **kw)["electron_budget"] == 4 and len(e.runs) > n


def test_given_ladders_are_kept(tmp_path, monkeypatch):
    e = Engine(lambda t, b, u, s: 1.0)
    best = _tune(e, tmp_path, monkeypatch, targets=(4096, 65536), budgets=(2, 8), turns=(3, -1), streams=(1, 2))
    assert best["event_target"] in (4096, 65536) and best["electron_budget"] in (2, 8)
    assert best["electron_turns"] in (3, -1) and best["streams"] in (1, 2)
    assert all(k == (0, 0, 0, 0) or k[0] in (4096, 65536) for k in e.runs)
