"""Run lists and powers of the protocol series (no GPU needed).

The run list must cover every step once, in order, and agree with the
waveform at each node of each step; the powers must equal step-by-step
products.
"""

import numpy as np
import pytest

from superspinsim_amd import configs, quadratures
from superspinsim_amd.protocol_runs import (
    RUN_DTYPE, ProtocolRuns, _padded, _times)
from superspinsim_amd.sweep import Waveform

H = 20e-12


def _waves(rng, count):
    out = []
    for _ in range(count):
        w = Waveform(5, base=[1.0, 0.0, 0.0, 0.0, 0.1])
        t = np.sort(rng.uniform(0, 60, 6)) * H
        t[1] = 7 * H                       # an edge on a step's start
        t = np.sort(t)
        w.add(1, t[0], t[1], 2.0, 3e9, 0.1)
        w.add(1, t[2], t[3], 1.0, 3e9)
        w.add(4, t[1], t[4], 0.5, 0.0, 0.0)
        if rng.random() < 0.5:
            w.add(4, t[4], np.inf, -0.3)
        out.append(w)
    return out


@pytest.mark.parametrize("scheme", [1, 2])
def test_runs_agree_with_the_waveforms(scheme):
    rng = np.random.default_rng(scheme)
    waves = _waves(rng, 12)
    nodes, _, _ = quadratures.scheme(scheme)
    steps = rng.integers(0, 70, 12)
    steps[3] = 0
    read_from = rng.integers(0, 60, 12)
    segs = {g: _padded(waves, g) for g in (1, 4)}
    base = np.array([w.base for w in waves])
    first, count, read, values, driven, inst = ProtocolRuns._layout(
        segs, base, 1, [4], nodes, steps, read_from, H)
    for i, w in enumerate(waves):
        mine = np.flatnonzero(inst == i)
        covered = [k for r in mine for k in range(first[r],
                                                  first[r] + count[r])]
        assert covered == list(range(steps[i]))
        for r in mine:
            for k in range(first[r], first[r] + count[r]):
                assert read[r] == (k >= read_from[i])
                on = False
                for s, c in enumerate(nodes):
                    at = w(float(_times(k, H, c)))
                    assert at[4] == values[r, s, 0]
                    on |= at[1] != 0
                assert driven[r] or not on
    # undriven runs exist, and steps split between the nodes (two nodes)
    assert np.any(~driven)
    assert np.any(np.ptp(values[:, :, 0], axis=1) != 0) == (scheme == 2)


def test_powers_equal_steps():
    wl = configs.odmr7(1, use_incoherent=True)
    const = wl.generators[0] + wl.excitation * wl.generators[4]
    n = wl.n
    powers = list(ProtocolRuns._powers([(const, H)], n, H, 9))
    step = np.eye(n) + powers[0][0]
    x0 = np.random.default_rng(0).standard_normal(n)
    x, xint = x0.copy(), np.zeros(n)
    for k in range(256):
        after = x + powers[0][0] @ x
        xint += 0.5 * H * (x + after)
        x = after
    d, read = powers[8]
    # rounding of 256 steps, half an ulp each
    assert np.max(np.abs(x0 + d @ x0 - x)) < 256 * 1.2e-16 * np.abs(x).max()
    assert np.max(np.abs(read @ x0 - xint)) < \
        256 * 1.2e-16 * np.abs(xint).max()
    assert np.max(np.abs(step @ step - np.eye(n) - powers[1][0])) < 1e-15


def test_cut_runs_end_after_the_steps_asked_for():
    rng = np.random.default_rng(5)
    waves = _waves(rng, 9)
    nodes, _, _ = quadratures.scheme(2)
    steps = rng.integers(20, 70, 9)
    segs = {g: _padded(waves, g) for g in (1, 4)}
    base = np.array([w.base for w in waves])
    first, count, read, _, _, inst = ProtocolRuns._layout(
        segs, base, 1, [4], nodes, steps, np.zeros(9, np.int64), H)
    rec = np.zeros(first.size, dtype=RUN_DTYPE)
    rec["first"], rec["count"], rec["read"] = first, count, read
    some = np.minimum(steps, rng.integers(0, 60, 9))
    some[4] = 0
    cut = ProtocolRuns.cut_records(rec, inst, some)
    assert np.array_equal(np.bincount(inst, cut["count"], 9), some)
    for k in range(9):
        end = 0
        for r in cut[(inst == k) & (cut["count"] > 0)]:
            assert r["first"] == end
            end += r["count"]
    assert np.array_equal(rec["count"], count)
    assert np.array_equal(cut[["first", "read"]], rec[["first", "read"]])


def test_tables_of_many_switch_values(monkeypatch):
    """As many tables as differ and are stepped through, each as its terms
    alone give it."""
    from superspinsim_amd import protocol_runs, series
    from superspinsim_amd.sweep import BatchSimulator
    monkeypatch.setattr(protocol_runs, "device_tensor", np.array)
    monkeypatch.setattr(ProtocolRuns, "_staged", staticmethod(np.copy))
    wl = configs.odmr7(1, use_incoherent=True)
    waves, steps = [], []
    for k in range(5):
        w = Waveform(5, base=[1.0, 0.0, 0.0, 0.0, 0.0])
        w.add(1, 0.0, 3.1e-10, 1e-4, 2e10)
        w.add(4, 5.05e-10, 9.4e-10, 0.01 * (k + 1))     # edges within steps
        waves.append(w)
        steps.append(60)
    sim = BatchSimulator(wl.generators, 2)
    _, const, program = sim.program(waves)
    runs = ProtocolRuns.build(sim, waves, const, program, np.array(steps),
                              np.zeros(5, np.int64), H,
                              lambda g: waves[0].abs_max()[g], 1e-16)
    table, rec = runs.d_table, runs.d_runs
    # the dark one, and per value one edge's pair (the other's swapped)
    assert len(np.unique(table.reshape(len(table), -1), axis=0)) == \
        len(table) == 11
    stepped = rec[rec["kind"] != protocol_runs.FREE]
    assert set(stepped["set0"]) | set(stepped["set1"]) == set(range(11))
    assert len(runs.d_powers) == 6
    alone = series.coefficient_matrices(
        [(sim.folded(const), 0.5 * H)], wl.generators[1], 7)
    driven = rec[rec["kind"] == protocol_runs.DRIVEN]
    assert np.unique(driven["set0"]).size == 1
    for k, m in enumerate(alone):
        assert np.array_equal(runs.model.sets[driven["set0"][0]][k], m)


@pytest.mark.parametrize("switched", [False, True])
def test_batch_of_no_steps(switched):
    """Protocols of no steps at all are left to the Taylor queue."""
    from superspinsim_amd.sweep import BatchSimulator
    wl = configs.odmr7(1, use_incoherent=True)
    w = Waveform(5, base=[1.0, 0.0, 0.0, 0.0, 0.0])
    w.add(1, 0.0, 1e-9, 1e-4, 2e10)
    if switched:
        w.add(4, 1e-9, 2e-9, 0.01)
    sim = BatchSimulator(wl.generators, 2)
    _, const, program = sim.program([w, w])
    assert ProtocolRuns.build(
        sim, [w, w], const, program, np.zeros(2, np.int64),
        np.zeros(2, np.int64), H, lambda g: w.abs_max()[g], 1e-16) is None
