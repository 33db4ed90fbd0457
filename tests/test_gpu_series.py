"""Series-in-the-drive kernel against the Taylor kernels (GPU).

Both propagate the same exponentials to 1e-16, so over the few thousand
exponentials of each case they differ by rounding only: at most one ulp of
the state per exponential, i.e. 4000 x 1.1e-16 = 4.4e-13 relative to the
largest value; 1e-12 is the bar.  ``taylor=17`` asks for the Taylor path on
every state.
"""

import importlib

import numpy as np
import pytest

from superspinsim_amd import configs
from superspinsim_amd.sweep import BatchSimulator, Waveform

pytestmark = pytest.mark.gpu

SAME = 1e-12


def _model(name):
    if name == "nv3":
        return configs.odmr3(1)
    return configs.odmr7(1, use_incoherent=name == "nv7c")


def _waves(wl, points, rabi, gated=False):
    b1 = configs.drive_amplitude(rabi)
    out = []
    for k in range(points):
        w = Waveform(5, base=[1.0, 0.0, 0.0, 0.0, wl.excitation])
        f = 2.80e9 + 1.4e8 * k / max(points - 1, 1)
        if gated:
            w.add(1, 1e-9, 5e-9 + 1e-10 * (k % 40), b1, 2 * np.pi * f, 0.3)
            w.add(1, 9e-9, 2e-8, -b1, 2 * np.pi * f, 0.1 * k)
        else:
            w.tone(1, b1, f)
        out.append(w)
    return out


@pytest.mark.parametrize("name,points,exps,fine,rabi,read,pack,orders", [
    ("nv7", 1, 2, 7, 3e6, "obs", True, (2, 1)),
    ("nv7", 5, 2, 16, 5e5, "integral", 3, (1, 1)),
    ("nv7", 4, 2, 33, 2.5e7, "full", 2, (2, 2)),
    ("nv7c", 7, 1, 20, 1.2e7, "full", 3, (2, 2)),
    ("nv7c", 2, 1, 50, 5e5, "obs", True, (1, 1)),
    ("nv3", 9, 2, 17, 5e6, "full", 7, (2, 1)),
    ("nv3", 15, 5, 11, 5e6, "obs", 7, (2, 1)),
    ("nv3", 3, 5, 10, 3e7, "integral", 2, (2, 2)),
    ("nv3", 3, 5, 10, 1e6, "integral", 2, (1, 1)),
    ("nv3", 3, 1, 10, 1e7, "obs", 5, (2, 2)),
    ("nv3", 65, 2, 10, 1e6, "obs", 7, (1, 1)),
])
def test_series_equals_taylor(gpu, name, points, exps, fine, rabi, read,
                              pack, orders):
    wl = _model(name)
    sim = BatchSimulator(wl.generators, exps, fine, pack=pack)
    dt = fine * 20e-12
    n_out = 1000 // fine
    args = (_waves(wl, points, rabi, gated=points > 4), wl.rho0, 3e-10,
            3e-10 + n_out * dt * (1 + 1e-9), dt)
    obs = None if read == "full" else wl.obs
    if points > 4 and obs is not None:
        obs = np.concatenate([obs, np.roll(obs, -1, axis=1)])
    print(f"{name} x {points}, {exps} exponentials, {read}", flush=True)
    got = sim.run(*args, obs=obs, read=read).cpu().numpy()
    assert sim.last_plan["series"] == orders, sim.last_plan
    want = sim.run(*args, obs=obs, read=read, taylor=17).cpu().numpy()
    assert got.shape == want.shape
    err = np.max(np.abs(got - want)) / np.max(np.abs(want))
    print(f"  {err:.1e}")
    assert err <= SAME


def test_every_state_and_own_initial_states(gpu):
    """Initial coherences everywhere: all 49 states in one wavefront, with a
    different state per instance; some sectors have no opposite."""
    wl = configs.odmr7(1)
    rng = np.random.default_rng(3)
    rho = rng.standard_normal((3, wl.n))
    sim = BatchSimulator(wl.generators, 2, 20)
    args = (_waves(wl, 3, 3e6), rho, 0.0, 20 * 4e-10 * (1 + 1e-9), 4e-10)
    got = sim.run(*args, read="full").cpu().numpy()
    assert sim.last_plan["involved"] == 49 and "series" in sim.last_plan
    want = sim.run(*args, read="full", taylor=17).cpu().numpy()
    assert np.max(np.abs(got - want)) / np.max(np.abs(want)) <= SAME


def test_undriven_run_and_non_finite_neighbour(gpu):
    """No driven generator at all; and an instance whose input is NaN leaves
    the instances that share its wavefront alone."""
    wl = configs.odmr7(1, use_incoherent=True)
    sim = BatchSimulator(wl.generators, 2, 10)
    free = [Waveform(5, base=[1.0, 0.0, 0.0, 0.0, wl.excitation])] * 3
    args = (0.0, 5 * 2e-10 * (1 + 1e-9), 2e-10)
    got = sim.run(free, wl.rho0, *args, read="full").cpu().numpy()
    assert "series" in sim.last_plan
    want = sim.run(free, wl.rho0, *args, read="full",
                   taylor=17).cpu().numpy()
    assert np.max(np.abs(got - want)) <= SAME
    rho = np.repeat(wl.rho0[None], 3, axis=0)
    rho[1, 2] = np.nan
    sim.pack = 3
    waves = _waves(wl, 3, 3e6)
    bad = sim.run(waves, rho, *args, obs=wl.obs).cpu().numpy()
    good = sim.run(waves, wl.rho0, *args, obs=wl.obs).cpu().numpy()
    assert np.all(np.isnan(bad[1])) and np.array_equal(bad[::2], good[::2])


def test_reduced_wide_states(gpu):
    """21 levels: the 171 involved states of 441, zeros elsewhere."""
    wl = configs.odmr21(2)
    sim = wl.simulator()
    waves = wl.waveforms()
    args = (waves, wl.rho0, 0.0, 2 * wl.time_step * (1 + 1e-9),
            wl.time_step)
    got = sim.run(*args, read="full").cpu().numpy()
    assert sim.last_plan["involved"] == 171
    want = sim.run(*args, read="full", taylor=11).cpu().numpy()
    assert np.max(np.abs(got - want)) / np.max(np.abs(want)) <= SAME
    obs = sim.run(*args, obs=wl.obs).cpu().numpy()[:, :, 0]
    assert np.max(np.abs(obs - got @ wl.obs[0])) <= 1e-15


def _protocols(seed, count, exps=2, early=False):
    """Pulses, waits and switched light with edges anywhere in a step; light
    and drive overlap in some."""
    wl = configs.odmr7(1, use_incoherent=seed % 2 == 1)
    rng = np.random.default_rng(seed)
    b1 = configs.drive_amplitude(3e6)
    waves, steps, read_from = [], [], []
    for k in range(count):
        w = Waveform(5, base=[1.0, 0.0, 0.0, 0.0,
                              0.01 if early else 0.0])
        t = np.cumsum(rng.uniform(0.05, 3.0, 6)) * 1e-9
        w.add(1, t[0], t[1], b1, 2 * np.pi * 2.87e9, 0.2)
        w.add(1, t[2], t[3], -b1, 2 * np.pi * 2.74e9, 0.0)
        w.add(4, t[3] - (0.5e-9 if k % 2 else 0.0), t[5],
              wl.excitation if k % 3 else 2 * wl.excitation)
        waves.append(w)
        steps.append(int(np.ceil(t[5] / 20e-12)) + 3 * (k % 2))
        read_from.append(int(t[2 + k % 3] / 20e-12))
    steps[0], read_from[1] = 0, steps[1] + 5
    batch = configs.ProtocolWorkload(
        "protocols", wl.generators, waves, wl.rho0, wl.obs, 20e-12,
        np.array(steps), np.array(read_from), {})
    return wl, batch, exps


@pytest.mark.parametrize("seed,count,exps,early", [
    (2, 7, 2, False), (3, 40, 2, True), (4, 5, 1, False)])
def test_protocol_runs_equal_steps(gpu, seed, count, exps, early):
    """Runs against the trapezoid of every step of a sweep through the Taylor
    kernel at degree 17 (at most 1,000 steps; a free run is at least as
    accurate as its steps)."""
    from superspinsim_amd.protocols import ProtocolBatch, trapezoid_window
    wl, pw, exps = _protocols(seed, count, exps, early)
    obs = np.concatenate([wl.obs, np.roll(wl.obs, 1, axis=1)])
    rng = np.random.default_rng(seed)
    rho = np.abs(rng.standard_normal((count, wl.n))) * (wl.rho0 != 0)
    b = ProtocolBatch(pw.generators, exps).prepare(
        pw.waves, rho, 20e-12, pw.steps, pw.read_from, obs)
    assert b.series is not None
    print(f"{count} protocols", flush=True)
    got = b.run().cpu().numpy().copy()
    last = int(pw.steps.max())
    trace = BatchSimulator(pw.generators, exps, 1).run(
        pw.waves, rho, 0.0, last * 20e-12 * (1 + 1e-12), 20e-12, obs=obs,
        taylor=17).cpu().numpy()
    assert trace.shape[1] == last
    want = np.stack([trapezoid_window(
        np.concatenate([(rho @ row)[:, None], trace[:, :, k]], axis=1),
        pw.read_from, pw.steps, 20e-12) for k, row in enumerate(obs)], axis=1)
    assert np.all(got[:2] == 0) and np.all(want[:2] == 0)
    err = np.max(np.abs(got - want)) / np.max(np.abs(want))
    print(f"  {err:.1e}")
    assert err <= SAME
    # without the counter
    b.out.fill_(np.nan)
    assert np.array_equal(b.launch_noalloc().cpu().numpy(), got)


@pytest.mark.parametrize("rotating,n,F,N,schemes", [
    (False, 3, 12, 30, 2), (True, 3, 12, 30, 5), (True, 4, 30, 7, 2),
    (False, 9, 7, 41, 3), (True, 19, 10, 20, 5), (False, 40, 50, 2, 1)])
def test_time_chunked_drop_in_equals_one_wavefront(gpu, monkeypatch,
                                                   rotating, n, F, N,
                                                   schemes):
    """One system cut in time against the same run on one wavefront: the
    chunk propagators hold n columns each, so the bar is that of the other
    comparisons times the chain's rounding (SAME x 4)."""
    gs = importlib.import_module("superspinsim_amd.generate_simulator")
    rng = np.random.default_rng(n)
    gens = rng.standard_normal((3, n, n)) * 1e9 / n
    gens[0] -= 2e9 * np.eye(n)
    kw = {}
    if rotating:
        nd = n // 2
        kw = dict(use_rotating=True, vectors_real=np.eye(n),
                  inv_vectors_real=np.eye(n),
                  doubles=np.stack([-rng.uniform(1e6, 1e8, nd),
                                    rng.uniform(-2e9, 2e9, nd)], axis=1),
                  singles=-rng.uniform(1e6, 1e7, n - 2 * nd))
        gens = gens[1:]

    def sampler(t, row):
        row[0] = np.cos(3e9 * t) if rotating else 1.0
        row[1] = np.sin(2e9 * t)
        if not rotating:
            row[2] = 0.3 * np.cos(1e9 * t)

    hil = 8                          # n rows of an 8 x 8 density
    vmap = np.array([(k // 8, k % 8, 0) if k // 8 <= k % 8 else
                     (k % 8, k // 8, 1) for k in range(n)])
    rho = rng.standard_normal((hil, hil))
    sim = gs.generate_simulator(sampler, gens, vmap,
                                number_of_exponentials=schemes,
                                number_of_fine_divisions=F, **kw)
    args = (rho, 1e-9, 1e-9 + N * F * 2e-11 * (1 + 1e-9), F * 2e-11)
    plans = []
    plan = gs.time_chunks
    monkeypatch.setattr(gs, "time_chunks", lambda *a, **k: (
        plans.append(plan(*a, **k)), plans[-1])[1])
    t1, got = sim(*args)
    assert plans and plans[0] is not None, plans
    monkeypatch.setattr(gs, "time_chunks", lambda *a, **k: None)
    t2, want = sim(*args)
    assert np.array_equal(t1, t2) and got.shape == want.shape
    err = np.max(np.abs(got - want)) / np.max(np.abs(want))
    print(f"n={n} chunks {plans[0]}: {err:.1e}", flush=True)
    assert err <= 4 * SAME


@pytest.mark.parametrize("name,exps,read", [
    ("nv3", 2, "full"), ("nv3", 5, "obs"), ("nv7c", 2, "obs")])
def test_chunked_series_equals_run(gpu, name, exps, read):
    wl = _model(name)
    sim = BatchSimulator(wl.generators, exps, 20)
    dt = 20 * 20e-12
    args = (_waves(wl, 3, 3e6), wl.rho0, 2e-9, 2e-9 + 50 * dt * (1 + 1e-9),
            dt)
    obs = None if read == "full" else wl.obs
    want = sim.run(*args, obs=obs, read=read).cpu().numpy()
    got = sim.run_chunked(*args, obs=obs, read=read, chunks=7).cpu().numpy()
    assert sim.last_plan["chunks"] == 7
    assert ("series" in sim.last_plan) == (exps == 2 or name == "nv3")
    err = np.max(np.abs(got - want)) / np.max(np.abs(want))
    print(f"{name}: {err:.1e}", flush=True)
    # node times counted from a chunk's start move by rounding: 4e-24 s in
    # phases of 2e10 rad/s, far below the state's own rounding
    assert err <= SAME


@pytest.mark.parametrize("name,points", [("nv7", 2100), ("nv21c", 3)])
def test_tables_outlive_a_launch_on_another_stream(gpu, name, points):
    """Tables staged on one stream, used on another, and dropped by the
    model for the next drive's before that launch has started."""
    import torch
    wl = configs.odmr21(1, use_incoherent=True) if name == "nv21c" else \
        _model(name)
    sim = BatchSimulator(wl.generators, 2, 10)
    args = (wl.rho0, 0.0, 3 * 2e-10 * (1 + 1e-9), 2e-10, wl.obs)
    first, next_ = (_waves(wl, points, rabi) for rabi in (3e5, 4e5))
    want = sim.run(first, *args).cpu().numpy()
    assert "series" in sim.last_plan
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        run = sim.prepare(first, *args)
        torch.cuda._sleep(50_000_000)
        run.launch()
    sizes = [t.numel() for t in vars(run).values()
             if isinstance(t, torch.Tensor) and t.dtype == torch.float64]
    rest = [t for k, t in vars(run).items()
            if k not in ("blocks", "columns", "table")]
    out = run.out
    del run
    sim.run(next_, *args)           # the model keeps these tables instead
    fill = [torch.full((n,), np.nan, dtype=torch.float64, device="cuda")
            for n in sizes for _ in range(4)]
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), want), (len(rest), len(fill))


def test_drop_in_without_room_for_chunks(gpu, monkeypatch):
    """Chunk propagators that cannot be allocated: one wavefront, the same
    states."""
    import torch
    gs = importlib.import_module("superspinsim_amd.generate_simulator")

    def sampler(t, row):
        row[0], row[1] = 1.0, np.sin(2e9 * t)

    rng = np.random.default_rng(1)
    gens = rng.standard_normal((2, 4, 4)) * 1e8 - 4e8 * np.eye(4)
    vmap = np.array([(0, 0, 0), (0, 1, 0), (0, 1, 1), (1, 1, 0)])
    sim = gs.generate_simulator(sampler, gens, vmap,
                                number_of_fine_divisions=30)
    args = (rng.standard_normal((2, 2)), 0.0, 20 * 6e-10, 6e-10)
    tried = []

    def full(*a, **kw):
        tried.append(1)
        raise torch.cuda.OutOfMemoryError("no room")

    monkeypatch.setattr(gs, "_chunked_states", full)
    got = sim(*args)[1]
    assert tried
    monkeypatch.setattr(gs, "time_chunks", lambda *a, **k: None)
    assert np.array_equal(got, sim(*args)[1])


@pytest.mark.parametrize("name,points,read", [
    ("nv7", 3, "full"), ("nv7", 2100, "obs"), ("nv3", 2100, "full"),
    ("nv21c", 3, "full")])
def test_launch_in_a_graph(gpu, name, points, read):
    """Every kernel's launch captured and replayed, with eager launches and
    another drive's tables between."""
    import torch
    wl = configs.odmr21(1, use_incoherent=True) if name == "nv21c" else \
        _model(name)
    sim = BatchSimulator(wl.generators, 2, 10)
    obs = None if read == "full" else wl.obs
    args = (wl.rho0, 0.0, 3 * 2e-10 * (1 + 1e-9), 2e-10, obs, read)
    first, next_ = (_waves(wl, points, rabi) for rabi in (3e5, 4e5))
    run = sim.prepare(first, *args)
    assert "series" in sim.last_plan
    want = run.launch().cpu().numpy().copy()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run.launch()
    for _ in range(3):
        sim.run(next_, *args)
        run.out.fill_(np.nan)
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(run.out.cpu().numpy(), want)
