"""Gradients of wide models through the series in the drive (GPU): the moment
and derivative kernels against numpy, whole gradients against the Frechet
chain (``store_inputs=False``)."""

import ctypes

import numpy as np
import pytest

from superspinsim_amd import _lib, configs
from superspinsim_amd.adjoint import GradientProblem
from superspinsim_amd.propagator import _ptr, device_tensor
from superspinsim_amd.series_gradient import derivative_matrices
from superspinsim_amd.series_wide_gradient import WideGradient
from superspinsim_amd.sweep import Waveform

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,points,exps,thetas,orders", [
    (65, 1, 2, 1, 4), (80, 9, 6, 2, 3), (81, 2, 40, 3, 4),
    (171, 2, 101, 12, 3), (171, 11, 10, 1, 4), (192, 1, 4, 1, 3)])
def test_moments_equal_numpy(gpu, n, points, exps, thetas, orders):
    """Sums of exps n^2 products in another order: exps n^2 / 2^53 of the sum
    of magnitudes at the very most, a thousandth of that in practice; the
    bar is 1e-13 of that sum.  The padding holds NaN."""
    import torch
    rng = np.random.default_rng(n)
    npad = -(-n // 16) * 16
    y, mu = np.full((2, points, exps, npad), np.nan)
    y[..., :n] = rng.standard_normal((points, exps, n))
    mu[..., :n] = rng.standard_normal((points, exps, n))
    f = rng.uniform(-1, 1, (points, exps))
    table = np.zeros((thetas, orders, npad, npad))
    table[:, :, :n, :n] = rng.standard_normal((thetas, orders, n, n))
    lib = _lib.load()
    work = torch.empty((points, lib.ssmx_series_moment_groups(n, orders),
                        thetas),
                       dtype=torch.float64, device="cuda")
    got = torch.empty((points, thetas), dtype=torch.float64, device="cuda")
    d = [device_tensor(a) for a in (y, mu, f, table)]
    _lib.check(lib.ssmx_series_moments(
        n, points, exps, orders, thetas, *[_ptr(a) for a in d], _ptr(work),
        _ptr(got), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    want, size = 0.0, 0.0
    for k in range(orders):
        m = np.einsum("pe,per,pec->prc", f ** k, mu[..., :n], y[..., :n])
        t = table[:, k, :n, :n]
        want = want + np.einsum("prc,trc->pt", m, t)
        size = size + np.einsum("prc,trc->pt", np.abs(m), np.abs(t))
    err = np.abs(got.cpu().numpy() - want) / size
    print(f"{err.max():.1e}")
    assert np.all(err <= 1e-13)


@pytest.mark.parametrize("n,thetas,orders", [(65, 1, 4), (171, 3, 4),
                                             (80, 2, 3)])
def test_derivatives_equal_numpy(gpu, n, thetas, orders):
    """The same recurrence in another order of summation: 1e-14 of each
    order's largest element.  f^3 is F^3 / 4 T_3(f / F) + 3 / 4 F^2 f."""
    rng = np.random.default_rng(n)
    far = np.abs(np.arange(n)[:, None] - np.arange(n)[None])
    a = rng.standard_normal((n, n)) * (far <= 3) * 0.05
    g = rng.standard_normal((n, n)) * (far == 4)
    da = rng.standard_normal((thetas, n, n)) * (far % 7 == 0)
    self = WideGradient()
    self.npad = -(-n // 16) * 16
    self.orders = orders
    got = self._derivatives(a, g, da, 30, 0.25).cpu().numpy()
    assert np.all(got[:, :, n:] == 0) and np.all(got[:, :, :, n:] == 0)
    want = derivative_matrices(a, g, da, 3)
    if orders == 3:
        want[1] += 0.75 * 0.25 ** 2 * want[3]
    for k in range(orders):
        err = np.max(np.abs(got[:, k, :n, :n] - want[k]))
        assert err <= 1e-14 * np.max(np.abs(want[k])), k


@pytest.mark.parametrize("points,outputs,fine,two,rabi", [
    (3, 5, 61, True, 0.5e6), (1, 1, 3, False, 0.5e6),
    (2, 2, 100, False, 0.5e6), (9, 3, 40, True, 3e6)])
def test_wide_gradient_equals_frechet(gpu, points, outputs, fine, two, rabi):
    """As for the 7-level models: each side is exact to its truncation
    relative to each exponential, a few 1e-12 of a gradient plus the
    cancellation floor 1e-12 F / theta_scale."""
    wl = configs.odmr21(1, use_incoherent=True)
    h = 20e-12
    b1 = configs.drive_amplitude(rabi)
    rng = np.random.default_rng(points)

    def waveforms(amps):
        out = []
        for f in np.linspace(2.868e9, 2.871e9, points):
            w = Waveform(5, base=[1.0, 0.0, 0.0, 0.0, wl.excitation])
            w.tone(1, b1, f)
            out.append(w)
        return out

    obs = wl.obs
    if two:
        obs = np.concatenate([obs, np.roll(obs, 1, axis=1)])
    rho = np.abs(rng.standard_normal(wl.n)) * (wl.rho0 != 0)
    theta = configs.nv21_theta0() * (1 + 0.01 * rng.standard_normal(12))
    seeds = rng.uniform(0.5, 1.5, (points, obs.shape[0]))
    res = {}
    for store in ("auto", False):
        problem = GradientProblem(
            lambda th: configs.nv21_generators(th, use_incoherent=True),
            waveforms, rho, obs, 1e-10,
            1e-10 + outputs * fine * h * (1 + 1e-9), fine * h, fine, 2, 300,
            adjoint_tolerance=1e-13 if not store else 1e-12,
            theta_scale=configs.THETA21_SCALE, store_inputs=store)
        out, state = problem.forward(theta, np.zeros(0))
        assert state["by_series"] == bool(store)
        back = problem.backward(state, seeds, lambda_out=True)
        res[bool(store)] = (out.cpu().numpy(),
                            {k: v.cpu().numpy() for k, v in back.items()})
    (fa, a), (fb, b) = res[True], res[False]
    assert np.max(np.abs(fa - fb)) <= 1e-12 * np.max(np.abs(fb))
    weight = (np.abs(fb) * seeds).sum(axis=1)
    err = np.abs(a["theta"] - b["theta"])
    floor = 1e-12 * weight[:, None] / configs.THETA21_SCALE[None]
    size = np.abs(b["theta"])
    print("theta", (err / (1e-11 * size + floor)).max(axis=0), flush=True)
    assert np.all(err <= 1e-11 * size + floor)
    e = np.max(np.abs(a["lambda"] - b["lambda"])) / \
        np.max(np.abs(b["lambda"]))
    assert e <= 1e-12


@pytest.mark.parametrize("steps", [3, 40])
def test_small_gradients_of_short_runs(gpu, steps):
    """Each parameter beside its own size, however small: the quadrupole's
    gradient hangs on entries of 1e-18 of the E_k over a few steps.  Against
    extended precision the Frechet chain is good to 4e-10 there."""
    wl = configs.odmr21(1, use_incoherent=True)
    b1 = configs.drive_amplitude(5e5)

    def waveforms(amps):
        w = Waveform(5, base=[1.0, 0.0, 0.0, 0.0, wl.excitation])
        w.tone(1, b1, 2.8695e9)
        return [w]

    res = {}
    for store in ("auto", False):
        problem = GradientProblem(
            lambda th: configs.nv21_generators(th, use_incoherent=True),
            waveforms, wl.rho0, wl.obs, 0.0, steps * 20e-12 * (1 + 1e-9),
            20e-12, 1, 2, 300, theta_scale=configs.THETA21_SCALE,
            store_inputs=store)
        out, state = problem.forward(configs.nv21_theta0(), [])
        assert state["by_series"] == bool(store)
        res[store] = problem.backward(state, np.ones((1, 1)))[
            "theta"].cpu().numpy()[0]
    names = np.array(configs.THETA21_NAMES)
    for name in ("D_gs", "radiative", "isc_pm", "quadrupole", "A_par",
                 "A_perp"):
        a, b = (r[names == name][0] for r in (res["auto"], res[False]))
        print(f"{name} {a / b - 1:.1e}", flush=True)
        assert abs(a / b - 1) <= 1e-9, name
