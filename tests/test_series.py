"""Series in the drive: tables and the choice of states (no GPU needed).

The E_k are compared with the whole exponent's Taylor series in extended
precision (scipy's expm is off by 2e-14 at the longer step), the omitted
orders with the plan's tolerance; ``reachable`` with brute-force
propagation; models the kernels do not cover must be refused.
"""

import ctypes
import os
import subprocess

import numpy as np
import pytest
from scipy.linalg import expm

from superspinsim_amd import _lib, configs, quadratures
from superspinsim_amd.series import (
    SeriesModel, coefficient_matrices, reachable, split_sectors)

H = 20e-12


def _pair(wl):
    return (wl.generators[0] + wl.excitation * wl.generators[4],
            wl.generators[1])


def _exponential(a):
    a = a.astype(np.longdouble)
    term = total = np.eye(a.shape[0], dtype=np.longdouble)
    for k in range(1, 60):
        term = term @ a / k
        total = total + term
    return total


@pytest.mark.parametrize("wl", [configs.odmr3(1),
                                configs.odmr7(1, use_incoherent=True)])
@pytest.mark.parametrize("scale", [H / 2, 2e-10])
def test_matrices_sum_to_the_exponential(wl, scale):
    const, drive = _pair(wl)
    mats = coefficient_matrices([(const, scale)], drive, 7)
    for f in (0.0, 1e-14, -wl.b1 * H):
        total = np.eye(wl.n) + sum(f ** k * m for k, m in enumerate(mats))
        want = _exponential(scale * const + f * drive)
        # rounding: a few ulp of the entries
        assert np.max(np.abs(total - want)) < 5e-15


@pytest.mark.parametrize("rabi,orders", [(5e5, (1, 1)), (3e6, (2, 1)),
                                         (2.5e7, (2, 2)), (1e9, None)])
def test_orders_meet_the_tolerance(rabi, orders):
    wl = configs.odmr7(1, use_incoherent=True)
    const, drive = _pair(wl)
    _, weights, _ = quadratures.scheme(2)
    model = SeriesModel.build(const, drive, weights, H)
    plan = model.plan(configs.drive_amplitude(rabi), 1e-16)
    assert (plan and plan[:2]) == orders
    if plan is None:
        return
    da, db, F = plan
    mats, = model.matrices(*plan)
    for f in F * np.linspace(-1, 1, 9):
        kept = np.eye(wl.n, dtype=np.longdouble) + sum(
            np.longdouble(f) ** k * m for k, m in enumerate(mats)
            if k <= (2 * da if k % 2 == 0 else 2 * db + 1))
        want = _exponential(H * weights[0].sum() * const + f * drive)
        # truncation 1e-16 / 8, and the tables' own rounding: half an ulp
        # of entries below 0.25 (1.4e-17 each, at most 11 in a column)
        assert np.abs(kept - want).sum(axis=0).max() <= 1.7e-16


def test_reachable_states_of_the_sweep():
    wl = configs.odmr7(1)
    const, drive = _pair(wl)
    pattern = (const != 0) | (drive != 0)
    states = reachable(pattern, wl.rho0[None], wl.obs)
    assert states.size == 19
    step = expm(H * const + wl.b1 * H * drive)
    x = np.linalg.matrix_power(step, 50) @ wl.rho0
    others = np.setdiff1d(np.arange(wl.n), states)
    assert np.all(x[others] == 0) and np.all(x[states] != 0)
    # a filled coherence brings its block in; a NaN counts as filled
    for value in (0.1, np.nan):
        rho = wl.rho0.copy()
        rho[others[0]] = value
        assert reachable(pattern, rho[None]).size > 19
    # nothing reaches the readout
    assert reachable(pattern, wl.rho0[None], np.zeros((1, wl.n))).size == 0


def test_uncovered_models_are_refused():
    _, weights, _ = quadratures.scheme(2)
    wl = configs.odmr7(1, use_incoherent=True)
    const, drive = _pair(wl)
    # a drive along the field couples within a sector
    assert SeriesModel.build(const, wl.generators[3], weights, H) is None
    # a transverse static field joins the sectors
    assert split_sectors(const + 1e-3 * drive, drive) is None
    # a long step
    assert SeriesModel.build(const, drive, weights, 1e-9) is None
    # five exponentials need three sets of tables
    _, w5, _ = quadratures.scheme(5)
    assert SeriesModel.build(const, drive, w5, H) is None
    _, w3, _ = quadratures.scheme(3)
    assert SeriesModel.build(const, drive, w3, H) is None
    small = _pair(configs.odmr3(1))
    assert len(SeriesModel.build(*small, w5, H).sets) == 3


def test_descriptor_layout_matches_header(tmp_path):
    include = os.path.join(os.path.dirname(os.path.dirname(
        os.path.abspath(__file__))), "include")
    (tmp_path / "p.c").write_text(r'''
#include <stddef.h>
#include <stdio.h>
#include "ssmx.h"
int main(void) {
  printf("%zu %zu %zu %zu\n", sizeof(ssmx_series_desc),
         offsetof(ssmx_series_desc, wave_group),
         offsetof(ssmx_series_desc, sector_rows),
         offsetof(ssmx_series_desc, h));
  return 0;
}
''')
    exe = str(tmp_path / "p")
    subprocess.run(["gcc", "-I", include, "-o", exe, str(tmp_path / "p.c")],
                   check=True)
    got = subprocess.run([exe], capture_output=True, text=True, check=True)
    D = _lib.SeriesDesc
    assert [int(v) for v in got.stdout.split()] == [
        ctypes.sizeof(D), D.wave_group.offset, D.sector_rows.offset,
        D.h.offset]


def test_derivative_matrices_match_differences():
    """Central differences of the extended-precision E_k with a step of
    1e-5: truncation of order 1e-10 of the entries."""
    from superspinsim_amd.series_gradient import derivative_matrices
    rng = np.random.default_rng(2)
    wl = configs.odmr3(1)
    const, drive = _pair(wl)
    const = const * (H / 2)
    dirs = rng.standard_normal((3,) + const.shape)
    got = derivative_matrices(const, drive, dirs, 5)
    for i, d in enumerate(dirs):
        up = coefficient_matrices([(const, 1.0), (d, 1e-5)], drive, 5, True)
        down = coefficient_matrices([(const, 1.0), (d, -1e-5)], drive, 5,
                                    True)
        for k in range(6):
            want = (up[k] - down[k]) / 2e-5
            assert np.max(np.abs(got[k, i] - want)) <= \
                1e-9 * np.max(np.abs(want))


def test_derivatives_between_sectors_the_drive_does_not_join(monkeypatch):
    """A parameter may couple two sectors that the drive leaves apart: its
    dE_0 is h dC to first order, in the lane of the column, at the row's
    slot of the opposite sector."""
    from superspinsim_amd import series, series_gradient
    from superspinsim_amd.sweep import BatchSimulator, Waveform
    for module in (series, series_gradient):
        monkeypatch.setattr(module, "device_tensor", np.asarray)
    const = np.diag([-1e8, -2e8, -3e8, -4e8])
    drive = np.zeros((4, 4))
    drive[2, 3] = drive[3, 2] = 1e9
    w = Waveform(2, base=[1.0, 0.0])
    w.tone(1, 1e-3, 1e9)
    sim = BatchSimulator(np.array([const, drive]), layout="plain")
    active, fixed, program = sim.program([w])
    dconst = np.zeros((1, 4, 4))
    dconst[0, 1, 0] = 1.0
    found = series_gradient.SeriesGradient.build(
        sim, fixed, program, [w], dconst, np.eye(4)[:1], np.eye(4)[1:2], H,
        1e-16, 1e-12)
    assert found is not None and found.n_theta == 1
    assert found.model.n_sectors == 2
    scale = H * sim.weights[0].sum()
    assert np.max(np.abs(found.d_dtable)) == pytest.approx(scale, rel=0.01)


@pytest.mark.parametrize("drive_max", [1e-95, 1e-148, 1e-155, 1e-300])
def test_negligible_drives_leave_finite_matrices(drive_max):
    """Powers of the largest drive that underflow, or whose inverse
    overflows: the kept orders are those of the power series."""
    from superspinsim_amd.series_gradient import SeriesGradient
    wl = configs.odmr7(1, use_incoherent=True)
    const, drive = _pair(wl)
    _, weights, _ = quadratures.scheme(2)
    model = SeriesModel.build(const, drive, weights, H)
    plan = model.plan(drive_max, 1e-16)
    assert plan is not None and plan[:2] == (1, 1)
    kept, = model.matrices(*plan)
    for k in range(4):
        assert np.array_equal(kept[k], model.sets[0][k]), k
    dmats = np.array(model.sets[0])[:, None]
    same = model.sector[:, None] == model.sector[None, :]
    for part, mats in zip((same, ~same), SeriesGradient._kept(
            dmats, plan[2], 1e-12, same)):
        for k, m in enumerate(mats):
            assert np.array_equal(m[0], model.sets[0][k] * part), k


@pytest.mark.parametrize("drive_max", [1e60, 1e300, np.inf])
def test_drives_beyond_the_number_range_are_refused(drive_max):
    """No plan (the Taylor path then refuses the run by its own error)."""
    from superspinsim_amd.series_wide import WideModel
    from superspinsim_amd.sweep import BatchSimulator, Waveform
    wl = configs.odmr7(1, use_incoherent=True)
    const, drive = _pair(wl)
    _, weights, _ = quadratures.scheme(2)
    model = SeriesModel.build(const, drive, weights, H)
    assert model.plan(drive_max, 1e-16) is None
    pairs = np.kron(np.eye(35), [[0.0, 1e9], [1e9, 0.0]])
    wide = WideModel.build(np.diag(np.full(70, -1e8)), pairs, weights, H)
    assert wide.plan(drive_max, 1e-16) is None
    w = Waveform(5, base=[1.0, 0.0, 0.0, 0.0, wl.excitation])
    w.tone(1, drive_max, 2.8e9)
    sim = BatchSimulator(wl.generators, 2, 20)
    point = sim.program([w])
    assert sim.series_plan([w], *point[1:], 4e-10) is None
    if np.isfinite(drive_max):
        with pytest.raises(ValueError, match="no Taylor plan"):
            sim.taylor_plan([w], *point, 4e-10)


def test_tables_of_two_drives_at_once(monkeypatch):
    """Another thread's drive between this one's tables being kept and
    returned: each gets its own."""
    from superspinsim_amd import series, series_wide
    monkeypatch.setattr(series, "device_tensor", np.asarray)
    monkeypatch.setattr(series_wide, "device_tensor", np.asarray)
    _, weights, _ = quadratures.scheme(2)
    wl = configs.odmr7(1, use_incoherent=True)
    pairs = np.kron(np.eye(35), [[0.0, 1e9], [1e9, 0.0]])

    def racing(base, kept, call):
        class Racing(base):
            def __setattr__(self, name, value):
                super().__setattr__(name, value)
                if name == kept and getattr(self, "other", None):
                    other, self.other = self.other, None
                    call(self, other)
        return Racing

    narrow = racing(SeriesModel, "_tables", lambda m, p: m.tables(*p))
    model = narrow.build(*_pair(wl), weights, H)
    plans = [model.plan(configs.drive_amplitude(r), 1e-16)
             for r in (5e5, 3e6)]
    model.other = plans[1]
    got = model.tables(*plans[0])
    assert model.other is None
    assert np.array_equal(got[1], SeriesModel.build(
        *_pair(wl), weights, H).tables(*plans[0])[1])

    wide = racing(series_wide.WideModel, "_layout",
                  lambda m, p: m.layout(p))
    args = np.diag(np.full(70, -1e8)), pairs, weights, H
    plans = [series_wide.WideModel.build(*args).plan(d, 1e-16)
             for d in (1e-7, 1e-5)]
    model = wide.build(*args)
    model.plan(1e-5, 1e-16)
    model._layout, model.other = None, plans[1]
    got = model.layout(plans[0])
    assert model.other is None
    assert np.array_equal(got[3], model._staged(
        model._arrays(*plans[0]))[3])


def test_reduced_simulator_follows_the_fine_divisions():
    from superspinsim_amd.sweep import BatchSimulator
    sim = BatchSimulator(configs.odmr7(1).generators, 2, 20)
    states = np.arange(5)
    assert sim._reduced(states).F == 20
    sim.F = 40
    assert sim._reduced(states).F == 40


def test_simulator_keeps_the_last_models():
    from superspinsim_amd import sweep
    wl = configs.odmr3(1)
    sim = sweep.BatchSimulator(wl.generators, 2, 20)

    def plan(k):
        w = sweep.Waveform(5, base=[1.0, 0.0, 0.0, 0.0, 1e-3 * (k + 1)])
        w.tone(1, wl.b1, 2.8e9)
        return sim.series_plan([w], *sim.program([w])[1:], 1e-9)[0]

    first = plan(0)
    second = plan(1)
    for k in range(2, sweep.MAX_MODELS):
        plan(k)
    assert plan(0) is first             # used again: stays
    plan(sweep.MAX_MODELS)
    assert len(sim._series_cache) == sweep.MAX_MODELS
    assert plan(0) is first and plan(1) is not second


def test_reach_covers_what_stays_within_it():
    from superspinsim_amd.series import Reach
    wl = configs.odmr7(1)
    const, drive = _pair(wl)
    reach = Reach((const != 0) | (drive != 0), wl.rho0[None], wl.obs)
    assert 0 < reach.states.size < wl.n
    rho = np.where(reach.ahead, 0.5, 0.0)[None]
    obs = np.where(reach.behind, 0.5, 0.0)[None]
    assert reach.covers(obs) and reach.covers(obs, rho)
    for k in np.flatnonzero(~reach.ahead):
        assert not reach.covers(obs, rho + np.eye(wl.n)[k])
    for k in np.flatnonzero(~reach.behind):
        assert not reach.covers(obs + np.eye(wl.n)[k])
    assert not reach.covers(obs, rho[:, 1:]) and not reach.covers(obs[:, 1:])


def test_gradient_store_that_cannot_be_had(monkeypatch):
    """Free memory in pieces: the checkpointed path, not an error."""
    import torch
    from superspinsim_amd import adjoint

    class Series:
        d_w = np.zeros((2, 2))
        store_shape = staticmethod(lambda *a: a)

    def empty(*args, **kw):
        raise torch.cuda.OutOfMemoryError("in pieces")

    problem = adjoint.GradientProblem(None, None, np.eye(4)[0], np.eye(4)[1],
                                      0.0, 1e-9, 1e-10)
    state = adjoint.GradientState(derivatives=True, n_inst=3)
    monkeypatch.setattr(adjoint, "_torch", lambda: torch)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda: (1 << 30,) * 2)
    for name in ("memory_reserved", "memory_allocated"):
        monkeypatch.setattr(torch.cuda, name, lambda: 0)
    monkeypatch.setattr(torch, "empty", empty)
    assert problem._series_store(state, Series, 10) is False
    assert problem._series_store(state, Series, 1 << 40) is False


@pytest.mark.parametrize("rabi", [5e5, 3e6])
def test_kept_derivatives_of_each_order_the_drive_brings(rabi):
    """What is cut off is small beside the lowest even and odd orders that a
    parameter can act through (1e-12), not only beside the whole: random
    directions within and between the sectors."""
    from superspinsim_amd.series_gradient import (
        SeriesGradient, derivative_matrices)
    wl = configs.odmr7(1, use_incoherent=True)
    const, drive = _pair(wl)
    _, weights, _ = quadratures.scheme(2)
    model = SeriesModel.build(const, drive, weights, H)
    F = model.plan(configs.drive_amplitude(rabi), 1e-16, 1e-12)[2]
    scale = H * weights[0].sum()
    same = model.sector[:, None] == model.sector[None, :]
    rng = np.random.default_rng(1)
    dirs = rng.standard_normal((4, wl.n, wl.n)) * 1e-3
    dirs[:2] *= same
    dirs[2:] *= ~same
    full = derivative_matrices(scale * const, drive, dirs, 9)
    kept = SeriesGradient._kept(full[:8], F, 1e-12, same)
    for f in F * np.array([1e-3, 0.3, -1.0]):
        for part, mats, even in ((same, kept[0], 2), (~same, kept[1], 0)):
            for odd, lead in ((0, even), (1, 1)):
                got = sum(f ** k * m for k, m in enumerate(mats)
                          if k % 2 == odd)
                want = sum(f ** k * m for k, m in enumerate(full)
                           if k % 2 == odd) * part
                for g, w, first in zip(got, want, full[lead] * part):
                    size = np.max(np.abs(F ** lead * first))
                    # (rounding of order 0, which may be far larger)
                    noise = 1e-15 * np.max(np.abs(w))
                    assert np.max(np.abs(g - w)) <= 1e-12 * size + noise
