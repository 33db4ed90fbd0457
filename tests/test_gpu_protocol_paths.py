"""Protocol batches by either path (GPU): the series in the drive (a batch
prepared without a Taylor plan) and the Taylor queue kernel (with one)."""

import numpy as np
import pytest

from superspinsim_amd import autotune, configs

pytestmark = pytest.mark.gpu

H = 20e-12
PATHS = [None, 11]


@pytest.fixture(scope="module")
def wl(gpu):
    return configs.pulsed7(count=24, seed=5, t_p_range=(2e-9, 20e-9),
                           tau_range=(10e-9, 100e-9), readout=50e-9)


def _batch(wl, taylor, steps=None, **kw):
    b = wl.batch().prepare(
        wl.waves, wl.rho0, H, wl.steps if steps is None else steps,
        wl.read_from, wl.obs, taylor=taylor, **kw)
    assert (b.series is None) == (taylor is not None)
    return b


@pytest.mark.parametrize("taylor", PATHS)
def test_tuning_trials_are_cut_and_paths_kept_apart(wl, taylor, tmp_path,
                                                    monkeypatch):
    monkeypatch.setenv("XDG_CACHE_HOME", str(tmp_path))
    b = _batch(wl, taylor)
    whole = b.run().cpu().numpy().copy()
    # what the trials launch: 2,000 steps of every protocol
    trials = []
    launch = b.launch
    monkeypatch.setattr(b, "launch", lambda *a, **k: (
        launch(*a, **k), trials.append(b.out.cpu().numpy().copy()))[0])
    choice = autotune.tune(b, trial_steps=2000, repeats=1)
    assert not choice["cached"] and choice["trial_steps"] == 2000
    plans = {(t["taylor"], t["substeps"]) for t in choice["trials"]}
    assert (len(plans) == 1) == (taylor is None)
    cut = _batch(wl, taylor, np.minimum(wl.steps, 2000)).run().cpu().numpy()
    assert 0 < np.count_nonzero(cut) < cut.size
    # (the Taylor trials have other degrees: 1e-10 as below)
    bar = 0.0 if taylor is None else 1e-10 * np.max(cut)
    assert trials and all(np.max(np.abs(t - cut)) <= bar for t in trials)
    got = b.run().cpu().numpy()
    assert np.max(np.abs(got - whole) / np.abs(whole)) < 1e-10
    # the choice holds for this path only
    assert autotune.tune(b, trial_steps=2000, repeats=1)["cached"]
    other = _batch(wl, 11 if taylor is None else None)
    assert not autotune.tune(other, trial_steps=2000, repeats=1)["cached"]


def test_cut_series_batch_equals_fewer_steps(wl):
    b = _batch(wl, None)
    whole = b.run().cpu().numpy().copy()
    steps = wl.steps - np.arange(len(wl.steps)) * 97
    b.series.cut(steps)
    got = b.run().cpu().numpy().copy()
    assert np.array_equal(got, _batch(wl, None, steps).run().cpu().numpy())
    b.series.cut()
    assert np.array_equal(b.run().cpu().numpy(), whole)


def _result(b):
    return b.out.cpu().numpy()[:, 0].copy()


@pytest.mark.parametrize("taylor", PATHS)
def test_grid_graph_and_stream_do_not_change_results(wl, taylor):
    import torch
    b = _batch(wl, taylor)
    want = b.run().cpu().numpy()[:, 0].copy()
    assert np.all(want != 0)
    for n_waves, wpb in ((1, 1), (5, 2), (7, 8)):
        got = _batch(wl, taylor, n_waves=n_waves, waves_per_block=wpb)
        got.run()
        assert np.array_equal(_result(got), want), (n_waves, wpb)
    b.out.fill_(np.nan)
    b.launch_noalloc()
    assert np.array_equal(_result(b), want)
    b.capture()
    scratch = torch.ones(1 << 20, dtype=torch.float64, device="cuda")
    for _ in range(3):
        scratch.mul_(1.5)               # unrelated eager work
        torch.cuda.synchronize()
        b.out.fill_(np.nan)
        b.graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(_result(b), want)
        assert int(b.counter.item()) == len(wl.waves) + b.n_waves
    side = torch.cuda.Stream()
    for _ in range(2):
        b.out.fill_(np.nan)
        side.wait_stream(torch.cuda.current_stream())
        b.launch(stream=side.cuda_stream)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        assert np.array_equal(_result(b), want)


def test_paths_agree_and_a_plan_set_later_changes_the_path(wl):
    """The Taylor plan set on a prepared series batch launches the Taylor
    queue; both within 1e-12 (9,355 steps, an ulp each at most)."""
    b = _batch(wl, None)
    series = b.run().cpu().numpy()[:, 0].copy()
    b.taylor = 13
    taylor = b.run().cpu().numpy()[:, 0].copy()
    assert np.array_equal(taylor, _batch(wl, 13).run().cpu().numpy()[:, 0])
    assert np.max(np.abs(series - taylor) / np.abs(taylor)) <= 1e-12
    b.taylor = b.plan_default[0]
    assert np.array_equal(b.run().cpu().numpy()[:, 0], series)


def test_protocols_of_no_steps(wl):
    from superspinsim_amd.protocols import ProtocolBatch
    none = np.zeros(len(wl.waves), dtype=np.int64)
    b = ProtocolBatch(wl.generators, 2).prepare(
        wl.waves, wl.rho0, H, none, none, wl.obs)
    b.out.fill_(np.nan)
    assert np.all(b.run().cpu().numpy() == 0)
