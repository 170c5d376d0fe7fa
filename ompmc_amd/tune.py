"""Autotuner of the event-queue form's launch parameters.

The batched form's queue knobs (``omc_run_opts``) are the particles in
flight per round (``event_target``), the electron steps between lane refills
(``electron_budget``), the refills an electron may hold its lane before it
is requeued (``electron_turns``) and the beamlet groups transported
concurrently (``streams``).  ``tune_dij`` searches them by coordinate
descent, timing settings on a sample of the caller's own beamlets at the
caller's photon splitting factor, and returns the fastest as keyword
arguments for ``Context.run_dij``, or the engine's automatic settings (0)
where nothing it tried is faster.  Results are cached per build, device and
workload shape in a JSON file, so a later process reuses them.  None of the knobs changes a
result beyond FP64 summation order: every history keeps its random-stream
key.

    from ompmc_amd import tune
    best = tune.tune_dij(ctx, phantom, spectrum, beamlets)
    ctx.run_dij(phantom, spectrum, beamlets, **best)
"""
from __future__ import annotations

import hashlib
import json
import os
import time

import numpy as np

from . import FORM_EVENT, FP32, LIB_PATH, event_defaults

CACHE = os.environ.get("OMC_TUNE_CACHE", os.path.join(os.path.expanduser("~"), ".cache", "ompmc_amd_tune.json"))

# Ladders of the knobs, to which the engine's defaults are added.  The search
# starts at these and moves along each ladder one rung at a time.
TARGETS = (262144, 524288, 1048576, 2097152, 4194304)     # four times that with photon splitting
BUDGETS = (2, 3, 4, 6, 8, 12, 16)
TURNS = (12, 18, 24, 30, 36, 48)
STREAMS = (1, 2, 3, 4)


def _sample(bix, n):
    from .phantoms import Beamlets
    sel = np.linspace(0, bix.n - 1, min(n, bix.n)).astype(int)
    return Beamlets(bix.ibeam[sel], bix.src, bix.corner[sel], bix.side1[sel], bix.side2[sel],
                    np.asarray(bix.nhist)[sel])


def _engine():
    """The build whose launches were timed: a digest of the library."""
    with open(LIB_PATH, "rb") as f:
        return hashlib.sha1(f.read()).hexdigest()[:12]


def _key(phantom, bix, precision, sample, nsplit, target):
    nvox = phantom.nreg - 1
    return (f"{_engine()}/target={target}/dij/{precision}/nvox={nvox}/beamlets={min(sample, bix.n)}/hist={int(np.median(bix.nhist))}"
            + (f"/nsplit={nsplit}" if nsplit > 1 else ""))


def _load():
    try:
        with open(CACHE) as f:
            return json.load(f)
    except (OSError, ValueError):
        return {}


def _store(d):
    try:
        os.makedirs(os.path.dirname(CACHE), exist_ok=True)
        with open(CACHE, "w") as f:
            json.dump(d, f, indent=1)
    except OSError:
        pass


def tune_dij(ctx, phantom, spectrum, bix, nbatch=10, precision=FP32, sample=200, targets=None, budgets=BUDGETS,
             turns=TURNS, streams=STREAMS, use_cache=True, verbose=False, nsplit=1, max_evals=24, margin=0.02):
    """Returns the fastest {event_target, electron_budget, electron_turns,
    streams} found (plus form, precision and nsplit) for ``Context.run_dij``
    on a sample of ``bix``, by coordinate descent: from the engine's defaults,
    each knob in turn tries the next rung up and down its ladder and moves while
    that is faster by more than ``margin`` (measurement noise), until no knob
    moves or ``max_evals`` settings have been timed.  Every setting computes
    the same matrix (the random streams do not depend on these knobs); only
    the time differs.  The engine's automatic settings, which depend on the
    run's groups, are timed as well unless the caller gives ladders, and
    returned (0 each) where the search finds nothing faster by more than
    ``margin``.  The default targets are four times larger with photon
    splitting, which carries nsplit times more electrons per history."""
    names = ("event_target", "electron_budget", "electron_turns", "streams")
    default = event_defaults(getattr(ctx, "device", 0), nsplit)
    key = _key(phantom, bix, precision, sample, nsplit, default["event_target"])
    cache = _load() if use_cache else {}
    if key in cache:
        return dict(cache[key]["opts"])
    automatic = targets is None and budgets is BUDGETS and turns is TURNS and streams is STREAMS
    ladders, pos = [], []
    for n, given, own in zip(names, (targets, budgets, turns, streams), (None, BUDGETS, TURNS, STREAMS)):
        if given is None:
            given = own = tuple(t * (4 if nsplit > 1 else 1) for t in TARGETS)
        ladder = sorted(set(given) | {default[n]}) if given is own else list(given)
        ladders.append(ladder)
        pos.append(ladder.index(default[n]) if default[n] in ladder else len(ladder) // 2)
    sub = _sample(bix, sample)
    ctx.run_dij(phantom, spectrum, sub, nbatch=nbatch, precision=precision, form=FORM_EVENT, nsplit=nsplit)
    timed = {}

    def rate_of(p):
        """Histories a second with the settings at rungs p (None: automatic)."""
        k = tuple(ladders[i][p[i]] for i in range(4)) if p else (0, 0, 0, 0)
        if k not in timed:
            kw = dict(zip(names, k))
            t0 = time.perf_counter()
            _, _, _, st = ctx.run_dij(phantom, spectrum, sub, nbatch=nbatch, precision=precision, form=FORM_EVENT,
                                      nsplit=nsplit, **kw)
            timed[k] = st.histories / (time.perf_counter() - t0)
            if verbose:
                print(f"tune: {kw}: {timed[k]:.4g} histories/s")
        return timed[k]

    auto = rate_of(None) if automatic else 0.0
    best = rate_of(pos)
    moved = True
    while moved and len(timed) < max_evals:
        moved = False
        for i in range(len(ladders)):
            for step in (1, -1):
                q = list(pos)
                q[i] += step
                if not 0 <= q[i] < len(ladders[i]) or len(timed) >= max_evals:
                    continue
                r = rate_of(q)
                if r > best * (1.0 + margin):
                    pos, best, moved = q, r, True
                    break
    if automatic and best <= auto * (1.0 + margin):
        best, knobs = auto, (0, 0, 0, 0)
    else:
        knobs = [ladders[i][pos[i]] for i in range(4)]
    opts = dict(form=FORM_EVENT, precision=precision, nsplit=nsplit, **dict(zip(names, knobs)))
    if use_cache:
        cache[key] = {"opts": opts, "histories_per_s": best,
                      "table": [dict(rate=r, **dict(zip(names, k))) for k, r in timed.items()]}
        _store(cache)
    return opts
