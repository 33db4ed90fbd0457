"""Gradients through the series in the drive against the Frechet chain (GPU).

``store_inputs=False`` takes the Taylor forward and the checkpointed Frechet
adjoint (degree 10, 1e-13 per exponential here); the default takes the
series. Both are exact to their truncation, which is relative to each
exponential: the parameter gradients differ by at most a few 1e-12 of their
own size plus the cancellation floor 1e-12 F / theta_scale that the oracle
comparison of the Frechet adjoint uses, over a thousand steps.
"""

import numpy as np
import pytest

from superspinsim_amd import configs
from superspinsim_amd.adjoint import GradientProblem
from superspinsim_amd.sweep import Waveform

pytestmark = pytest.mark.gpu


def _problem(exps, incoherent, points, outputs, fine, rabi, store, two_rows,
             seed=5):
    wl = configs.odmr7(1, use_incoherent=incoherent)
    rng = np.random.default_rng(seed)
    scale = configs.drive_amplitude(1.0)
    h = 20e-12 if exps == 2 else 10e-12
    end = outputs * fine * h
    # segments with gaps, an edge on a step, edges inside steps
    edges = np.array([0.0, 0.13, 0.2, 0.3703, 0.37045, 0.9]) * end
    edges[2] = round(0.2 * end / h) * h
    freqs = rng.uniform(2.70e9, 2.76e9, points)

    def waveforms(amps):
        out = []
        for f in freqs:
            w = Waveform(5, base=[1.0, 0.0, 0.0, 0.0, wl.excitation])
            for k, (a, b) in enumerate(((0, 1), (2, 3), (4, 5))):
                w.add(1, edges[a], edges[b], scale * amps[k],
                      2 * np.pi * f, 0.3 * k, param=k, dparam=scale)
            # an untagged segment between tagged ones
            w.add(1, edges[3], edges[4], scale * rabi, 2 * np.pi * f, 0.0)
            out.append(w)
        return out

    rho = np.array([1.0 if (y, x) == (1, 1) else 0.0
                    for y, x, _ in wl.vmap])
    obs = wl.obs
    if two_rows:
        obs = np.concatenate([obs, rho[None]])
    problem = GradientProblem(
        lambda th: configs.nv7_generators(th, use_incoherent=incoherent),
        waveforms, rho, obs, 1e-10, 1e-10 + end * (1 + 1e-9), fine * h, fine,
        exps, 300, adjoint_tolerance=1e-13 if not store else 1e-12,
        theta_scale=configs.THETA_SCALE,
        store_inputs=False if not store else "auto")
    theta = configs.nv7_theta0() * (1 + 0.01 * rng.standard_normal(9))
    amps = rng.normal(rabi, rabi / 6, 3)
    seeds = rng.uniform(0.5, 1.5, (points, obs.shape[0]))
    return problem, theta, amps, seeds


@pytest.mark.parametrize("exps,incoherent,points,outputs,fine,rabi,two", [
    (2, False, 3, 10, 100, 3e6, False), (2, True, 5, 7, 61, 8e6, True),
    (2, True, 1, 1, 3, 3e5, False), (1, True, 2, 30, 33, 3e6, False)])
def test_series_gradient_equals_frechet(gpu, exps, incoherent, points,
                                        outputs, fine, rabi, two):
    res = {}
    for store in (True, False):
        problem, theta, amps, seeds = _problem(
            exps, incoherent, points, outputs, fine, rabi, store, two)
        out, state = problem.forward(theta, amps)
        assert state["by_series"] == store
        back = problem.backward(state, seeds, lambda_out=True)
        res[store] = (out.cpu().numpy(),
                      {k: v.cpu().numpy() for k, v in back.items()})
    (fa, a), (fb, b) = res[True], res[False]
    assert np.max(np.abs(fa - fb)) <= 1e-12 * np.max(np.abs(fb))
    weight = (np.abs(fb) * seeds).sum(axis=1)
    err = np.abs(a["theta"] - b["theta"])
    floor = 1e-12 * weight[:, None] / configs.THETA_SCALE[None]
    size = np.abs(b["theta"])
    print("theta", (err / (1e-11 * size + floor)).max(axis=0), flush=True)
    assert np.all(err <= 1e-11 * size + floor)
    for key in ("records", "amplitudes"):
        # (all zero where three steps are too short for any effect)
        e, most = np.max(np.abs(a[key] - b[key])), np.max(np.abs(b[key]))
        print(key, f"{e:.1e} of {most:.1e}")
        assert e <= 1e-10 * most
    e = np.max(np.abs(a["lambda"] - b["lambda"])) / \
        np.max(np.abs(b["lambda"]))
    assert e <= 1e-12


def test_parameter_that_joins_what_the_drive_does_not(gpu):
    """State 1, which is read, gets theta times state 0: at theta = 0 its
    derivative is (exp(-a t) - exp(-b t)) / (b - a), summed by the
    trapezoid rule as the readout.  The truncation of an exponential's
    derivative, 1e-12 of it, adds up over the exponentials a state has seen:
    a weighted mean of them, so the bar is 1e-12 with the rounding of 1,000
    steps (1e-13) below it."""
    a, b, h, steps = 1e8, 3e8, 20e-12, 1000
    drive = np.zeros((4, 4))
    drive[2, 3] = drive[3, 2] = 1e9

    def generators(theta):
        const = np.diag([-a, -b, -1e8, -2e8])
        const[1, 0] = theta[0]
        return np.array([const, drive])

    def waveforms(amps):
        w = Waveform(2, base=[1.0, 0.0])
        w.tone(1, 1e-3, 1e9)
        return [w, w]

    problem = GradientProblem(
        generators, waveforms, np.eye(4)[0], np.eye(4)[1], 0.0,
        steps * h * (1 + 1e-9), 10 * h, 10, 2, theta_scale=[1e8])
    out, state = problem.forward([0.0], [])
    assert state["by_series"] and state["series"].model.n == 2
    got = problem.backward(state, np.ones((2, 1)))["theta"].cpu().numpy()
    t = h * np.arange(steps + 1)
    s = (np.exp(-a * t) - np.exp(-b * t)) / (b - a)
    want = 0.5 * h * np.sum(s[:-1] + s[1:])
    print(f"{np.max(np.abs(got / want - 1)):.1e}", flush=True)
    assert np.all(out.cpu().numpy() == 0)
    assert np.max(np.abs(got / want - 1)) <= 1e-12


def test_states_and_rows_set_after_setup(gpu):
    """A point set up for one initial state and readout serves any other,
    through the Taylor path where they involve further states: as a point
    set up for them, to the bars above."""
    problem, theta, amps, seeds = _problem(2, False, 2, 4, 20, 3e6, True,
                                           False)
    n = problem.rho0.size
    state = problem.setup(theta, amps)
    out, _ = problem.forward(theta, amps, state)
    assert state["by_series"]
    first = out.cpu().numpy().copy()
    reach = state["series"].reach
    rng = np.random.default_rng(0)
    rho, obs = rng.standard_normal((2, n))
    rho[reach.ahead], obs[reach.behind] = problem.rho0[reach.ahead], 0.3

    def gradients(st):
        out, st = problem.forward(theta, amps, st)
        back = problem.backward(st, seeds, lambda_out=True)
        return out.cpu().numpy(), [back[k].cpu().numpy() for k in (
            "theta", "amplitudes", "lambda")], st["by_series"]

    saved = problem.rho0, problem.obs
    for new in ((rho, saved[1]), (saved[0], obs[None]), (rho, obs[None])):
        problem.rho0, problem.obs = new
        got = gradients(state)
        want = gradients(problem.setup(theta, amps))
        assert not got[2]
        assert np.max(np.abs(got[0] - want[0])) <= \
            1e-12 * np.max(np.abs(want[0]))
        for a, b in zip(got[1], want[1]):
            size = np.max(np.abs(b), axis=0) if a.ndim == 2 else \
                np.max(np.abs(b))
            assert np.all(np.abs(a - b) <= 1e-10 * size + 1e-300)
    # rows set between the two directions
    problem.rho0, problem.obs = saved
    out, _ = problem.forward(theta, amps, state)
    assert state["by_series"] and np.array_equal(out.cpu().numpy(), first)
    problem.obs = obs[None]
    got = problem.backward(state, seeds)["theta"].cpu().numpy()
    want = gradients(problem.setup(theta, amps))[1][0]
    assert np.all(np.abs(got - want) <= 1e-10 * np.max(np.abs(want), axis=0))


@pytest.mark.parametrize("steps,b", [(3, 1.5e-4), (50, 1.5e-4), (3, 1.5e-3),
                                     (50, 5e-6)])
def test_amplitude_gradient_of_a_weak_rotation(gpu, steps, b):
    """Two states that a constant drive rotates into each other, both
    decaying: the read one is exp(-a t) cos(g c t), its derivative in c
    -g t exp(-a t) sin(g c t), of second order in the drive.  1e-12 as
    asked for, of the derivative itself (b is half a step's angle)."""
    a, h, g = 1e8, 20e-12, 1e9
    c = b / (0.5 * h * g)
    drive = np.array([[0.0, -g], [g, 0.0]])

    def waveforms(amps):
        w = Waveform(2, base=[1.0, 0.0])
        w.add(1, 0.0, 1.0, amps[0], param=0, dparam=1.0)
        return [w, w, w]

    problem = GradientProblem(
        lambda th: np.array([np.diag([-a, -a]), drive]), waveforms,
        np.eye(2)[0], np.eye(2)[0], 0.0, steps * h * (1 + 1e-9), h, 1, 2)
    out, state = problem.forward([], [c])
    assert state["by_series"]
    got = problem.backward(state, np.ones((3, 1)))["amplitudes"].cpu().numpy()
    t = h * np.arange(steps + 1)
    s = -3 * g * t * np.exp(-a * t) * np.sin(g * c * t)
    want = 0.5 * h * np.sum(s[:-1] + s[1:])
    print(f"{got[0] / want - 1:.1e}", flush=True)
    assert abs(got[0] / want - 1) <= 1e-12
