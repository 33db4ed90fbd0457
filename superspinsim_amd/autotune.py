"""Autotuner for the persistent protocol launches.

Chooses, by measurement on the device, the launch shape (wavefronts per
workgroup) and the Taylor plan of a ``ProtocolBatch``:

* every candidate plan meets the same truncation bound (the propagator's
  measured plan at the batch tolerance), so the choice changes speed, not
  accuracy: degree m with s = 1, 2, 4 substeps, i.e. the exponent norm above
  which an exponential is split into 2^k parts;
* wavefronts per workgroup 1, 2, 4 or 8 (generator values are staged once
  per workgroup in LDS; more wavefronts share one copy).

A batch that runs as series in the drive (``ProtocolBatch.series``) has no
Taylor plan to choose: only the wavefronts per workgroup are tried.

Each candidate runs on a trial copy of the batch: its longest instances (one
grid's worth), truncated to ``trial_steps`` steps, timed with HIP events on
the launch stream.  Results are cached per device, path and problem shape in
``$XDG_CACHE_HOME/superspinsim_amd/autotune.json`` (default ``~/.cache``).
"""

import json
import os

import numpy as np

from superspinsim_amd import _lib
from superspinsim_amd.propagator import _torch, taylor_plan_measured

WAVES_PER_BLOCK = (1, 2, 4, 8)
SUBSTEPS = (1, 2, 4)


def cache_path():
    root = os.environ.get("XDG_CACHE_HOME") or os.path.join(
        os.path.expanduser("~"), ".cache")
    return os.path.join(root, "superspinsim_amd", "autotune.json")


def _load_cache():
    try:
        with open(cache_path()) as f:
            return json.load(f)
    except (OSError, ValueError):
        return {}


def _store_cache(cache):
    path = cache_path()
    try:
        os.makedirs(os.path.dirname(path), exist_ok=True)
        tmp = path + ".tmp"
        with open(tmp, "w") as f:
            json.dump(cache, f, indent=1, sort_keys=True)
        os.replace(tmp, path)
    except OSError:
        pass                            # a read-only home only loses caching


def plan_candidates(batch, samples):
    """(m, s) plans meeting the batch tolerance for s in SUBSTEPS."""
    prop = batch.prop
    exps = prop.sample_exponents(samples, batch.h)
    out = []
    for s in SUBSTEPS:
        try:
            # the measured plan restricted to exactly s substeps
            scaled = [a / s for a in exps]
            m, _ = taylor_plan_measured(scaled, tol=batch.tolerance / s,
                                        max_substeps=1)
        except ValueError:
            continue
        if (m, s) not in out:
            out.append((m, s))
    return out


def problem_key(batch):
    """Cache key: the device, the path (a choice made for one kernel says
    nothing about the other) and the problem's shape."""
    name = _torch().cuda.get_device_properties(0).name
    if batch.series is not None:
        model, plan = batch.series.model, batch.series.plan
        J, S = batch.sim.weights.shape
        shape = ("series", model.n, plan[0], plan[1], len(model.sets), J, S)
    else:
        prop = batch.prop
        shape = ("taylor", prop.n, prop.ell.slots, prop.K, prop.J, prop.S,
                 prop.ell.nnz)
    return "|".join(str(v) for v in (name,) + shape + (
        batch.tolerance, batch.n_obs))


def tune(batch, trial_steps=20000, repeats=2, use_cache=True, verbose=False):
    """Measure every candidate on a trial copy; apply and return the best.

    Returns a dict with the chosen ``waves_per_block``, ``taylor``,
    ``substeps``, the per-candidate times (ms) and whether it came from the
    cache.
    """
    torch = _torch()
    cache = _load_cache() if use_cache else {}
    key = problem_key(batch)
    if batch.series is not None:
        # runs of the series in the drive: only the grid's shape is open
        plans = [tuple(batch.plan_default)]
    else:
        plans = plan_candidates(batch, batch.sim.coefficient_box(
            batch.waves_host, batch.program))
    if use_cache and key in cache:
        best = cache[key]
        if (best["taylor"], best["substeps"]) in [tuple(p) for p in plans]:
            apply(batch, best)
            return dict(best, cached=True)

    # trial copy: the longest instances, one grid's worth, truncated
    saved = (batch.steps.copy(), batch.read_from.copy(), batch.n_waves,
             batch.waves_per_block, batch.taylor, batch.substeps)
    count = min(batch.n_inst, batch.n_waves)
    trial_steps_arr = np.minimum(batch.steps, trial_steps)
    trial_read = np.minimum(batch.read_from, trial_steps_arr)
    order = batch.order[:count]
    mask = np.zeros(batch.n_inst, dtype=bool)
    mask[order] = True
    trial_steps_arr = np.where(mask, trial_steps_arr, 0)
    batch.d_steps.copy_(torch.from_numpy(trial_steps_arr))
    batch.d_read_from.copy_(torch.from_numpy(trial_read))
    if batch.series is not None:
        batch.series.cut(trial_steps_arr)
    results = []
    try:
        for m, s in plans:
            for wpb in WAVES_PER_BLOCK:
                batch.taylor, batch.substeps = m, s
                batch.waves_per_block = wpb
                batch.launch()              # warm
                stream = torch.cuda.current_stream()
                ev = [torch.cuda.Event(enable_timing=True)
                      for _ in range(2)]
                ev[0].record(stream)
                for _ in range(repeats):
                    batch.launch()
                ev[1].record(stream)
                torch.cuda.synchronize()
                ms = ev[0].elapsed_time(ev[1]) / repeats
                results.append(dict(taylor=m, substeps=s,
                                    waves_per_block=wpb, ms=ms))
                if verbose:
                    print(f"tune: m={m} s={s} wpb={wpb}: {ms:.3f} ms")
    finally:
        steps, read_from, n_waves, wpb, m, s = saved
        batch.d_steps.copy_(torch.from_numpy(steps))
        batch.d_read_from.copy_(torch.from_numpy(read_from))
        batch.n_waves, batch.waves_per_block = n_waves, wpb
        batch.taylor, batch.substeps = m, s
        torch.cuda.synchronize()
        if batch.series is not None:
            batch.series.cut()
    best = min(results, key=lambda r: r["ms"])
    choice = dict(waves_per_block=best["waves_per_block"],
                  taylor=best["taylor"], substeps=best["substeps"],
                  trial_steps=int(trial_steps), trials=results)
    if use_cache:
        cache[key] = choice
        _store_cache(cache)
    apply(batch, choice)
    return dict(choice, cached=False)


def apply(batch, choice):
    batch.waves_per_block = int(choice["waves_per_block"])
    batch.taylor = int(choice["taylor"])
    batch.substeps = int(choice["substeps"])
    if not 1 <= batch.taylor <= _lib.MAX_TAYLOR:
        raise ValueError("tuned Taylor degree out of range")


__all__ = ["tune", "plan_candidates", "cache_path", "apply"]
