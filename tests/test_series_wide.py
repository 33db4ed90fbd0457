"""The series in the drive above a wavefront's rows: layout on the CPU, kernel
against the Taylor kernels on the GPU.

``_model(n, block)``: blocks of ``block`` states in two halves, a constant
part within the halves and a drive across; couplings reach 14 states far and
E_k is dense within the blocks.  With ``spread`` a first few rows depend on
every block as well.  Rows stay within the 32 columns of the Taylor kernels.
"""

import numpy as np
import pytest

from superspinsim_amd import configs, quadratures, series_wide
from superspinsim_amd.series import coefficient_matrices
from superspinsim_amd.series_wide import WideModel, wide_coefficients
from superspinsim_amd.sweep import BatchSimulator, Waveform

H = 2e-11


def _model(n, block, norm=0.15, spread=0):
    rng = np.random.default_rng(n)
    place = np.arange(n)
    same = place[:, None] // block == place[None, :] // block
    half = (place % block) % 2
    near = np.abs(place[:, None] - place[None, :]) <= 14
    same[:spread] = True
    near[:spread, ::11] = True
    same &= near
    inner = same & (half[:, None] == half[None, :])
    const = rng.standard_normal((n, n)) * inner
    const -= np.diag(np.abs(const).sum(axis=0))
    const *= norm / (0.5 * H * np.abs(const).sum(axis=0).max())
    drive = rng.standard_normal((n, n))
    drive = (drive - drive.T) * (same & ~inner)
    return const, drive / np.abs(drive).sum(axis=0).max()


@pytest.mark.parametrize("n,block,spread,lanes,slots,amp,orders", [
    (65, 65, 0, 8, 5, 1e7, (1, 1)), (112, 112, 0, 8, 7, 1e7, (1, 1)),
    (150, 10, 3, 16, 5, 1e7, (1, 1)), (192, 8, 0, 8, 4, 1e7, (1, 1)),
    (112, 112, 0, 8, 7, 1e8, (2, 1)), (65, 65, 0, 8, 5, 5e8, (2, 2)),
    (150, 10, 3, 16, 5, 5e8, (2, 2)), (120, 120, 0, 8, 8, 1e8, (2, 1))])
def test_layout_holds_the_matrices(monkeypatch, n, block, spread, lanes,
                                   slots, amp, orders):
    monkeypatch.setattr(series_wide, "device_tensor", lambda a: a)
    const, drive = _model(n, block, spread=spread)
    _, weights, _ = quadratures.scheme(2)
    model = WideModel.build(const, drive, weights, H)
    plan = model.plan(amp, 1e-16)
    F = plan[2]
    assert plan[:2] == orders
    high = sum(orders) - 2
    blocks, states, columns, table, in_lds = model.layout(plan)
    assert tuple(blocks[0, :2]) == (slots, lanes)
    assert in_lds == sum(high * s + 4 * max(0, s - 7)
                         for s in blocks[:, 0])
    kept = [np.zeros((n, n)) for _ in range(6)]
    where = {int(p): int(s) for p, s in states.reshape(-1, 2) if p >= 0}
    assert sorted(where.values()) == list(range(n))
    for w, (c, width, at, tat) in enumerate(blocks):
        col = columns[at:at + 2 * c * 64].reshape(2 * c, 64)
        r = min(c, 7)
        held = table[tat:tat + 2 * r * 256].reshape(2, r, 4, 64)
        tat += 2 * r * 256
        hi = table[tat:][:high * c * 128].reshape(high * c, 64, 2)
        tat += high * c * 128
        rest = table[tat:][:(c - r) * 512].reshape(c - r, 2, 2, 64, 2)
        tab = np.concatenate([np.concatenate([held[part], rest[
            :, part].transpose(0, 1, 3, 2).reshape(c - r, 4, 64)])
            for part in (0, 1)])
        for lane in range(64):
            first = lane % 32 - lane % 32 % (width // 2)
            for i in (0, 1):
                p, row = states[w, first + 32 * i]
                for e in range(2 * c):
                    for o in (0, 1):
                        if tab[e, 2 * o + i, lane] != 0.0:
                            kept[2 * o + e // c][row, where[
                                int(col[e, lane])]] += tab[e, 2 * o + i,
                                                           lane]
                    if e < high * c:
                        kept[4 + e // c][row, where[int(col[e, lane])]] += \
                            hi[e, lane, i]
                if p < 0:
                    assert not np.any(tab[:, i::2, lane])
                    assert not np.any(hi[:, lane, i])
    # against the whole series at the ends and inside: what is left out
    # stays below the tolerance (half an ulp of the sums' largest
    # coefficient, 0.15, on top: 1.4e-17 per entry, n / 2 of them a column)
    whole = coefficient_matrices([(const, 0.5 * H)], drive, 9, extended=True)
    for f in (0.0, 0.37 * F, -F):
        got = sum(np.longdouble(f) ** k * m for k, m in enumerate(kept))
        want = sum(np.longdouble(f) ** k * m for k, m in enumerate(whole))
        err = np.abs(got - want).sum(axis=0).max()
        assert err <= 1e-16 + 1.4e-17 * n / 2


def test_coefficients_in_doubles_from_degree_three():
    """Terms of degree three on are (1/4)^3 / 6 at most: ten ulp of theirs
    are 2e-17 / 4, a tenth of the ulp of a quarter."""
    const, drive = _model(70, 70, norm=0.25)
    got = wide_coefficients([(const, 0.5 * H)], drive, 4)
    want = coefficient_matrices([(const, 0.5 * H)], drive, 4)
    for k in range(3):
        scale = np.max(np.abs(want[k]))
        assert np.max(np.abs(got[k] - want[k])) <= 2.3e-16 * scale


def test_uncovered_models_are_refused(monkeypatch):
    monkeypatch.setattr(series_wide, "device_tensor", lambda a: a)
    _, weights, _ = quadratures.scheme(2)
    # 64 rows, 257 rows, one exponential
    for n, exps in ((64, 2), (257, 2), (70, 1)):
        w = quadratures.scheme(exps)[1]
        assert WideModel.build(*_model(n, 10), w, H) is None
    # more pairs than the wavefronts hold; rows of more columns than the
    # lanes; a drive so large that order six counts; rows whose orders above
    # three exceed the LDS
    for n, block, amp in ((193, 8, 1e7), (190, 190, 1e7), (70, 70, 1e10),
                          (192, 100, 5e8)):
        model = WideModel.build(*_model(n, block), weights, H)
        assert model.plan(amp, 1e-16) is None
    const, drive = _model(70, 10)
    assert WideModel.build(const, drive + const, weights, H) is None
    assert WideModel.build(100 * const, drive, weights, H) is None


@pytest.mark.gpu
@pytest.mark.parametrize("n,block,spread,norm,points,fine,read,scale,orders", [
    (65, 65, 0, 0.15, 1, 7, "obs", 1, (1, 1)),
    (112, 112, 0, 0.9, 3, 33, "full", 1, (1, 1)),
    (150, 10, 3, 0.15, 5, 1, "integral", 1, (1, 1)),
    (192, 8, 0, 0.15, 2, 40, "obs", 1, (1, 1)),
    (171, 0, 0, 0.0, 3, 16, "integral", 1, (1, 1)),
    (441, 0, 0, 0.0, 2, 31, "full", 1, (1, 1)),
    (112, 112, 0, 0.15, 3, 20, "obs", 10, (2, 1)),
    (150, 10, 3, 0.15, 2, 33, "integral", 50, (2, 2)),
    (120, 120, 0, 0.15, 2, 9, "full", 1, (1, 1)),
    (171, 0, 0, 0.0, 2, 16, "obs", 6, (2, 1)),
    (65, 65, 0, 0.15, 3, 21, "full", 50, (2, 2))])
def test_wide_series_equals_taylor(gpu, n, block, spread, norm, points, fine,
                                   read, scale, orders):
    """Both propagate the same exponentials to 1e-16; over 600 steps they
    differ by rounding, an ulp of the state per exponential at most
    (1200 x 1.1e-16 = 1.3e-13, times the few units by which the random
    models amplify): 1e-12."""
    if block:
        const, drive = _model(n, block, norm, spread)
        gens = np.stack([const, drive])
        rng = np.random.default_rng(1)
        rho = rng.standard_normal((points, n))
        obs = rng.standard_normal((2, n))
        base, f0, amp = [1.0, 0.0], 2.87e9, 1e7
    else:
        wl = configs.odmr21(1, use_incoherent=n == 171)
        gens, rho, obs = wl.generators, wl.rho0, wl.obs
        base = [1.0, 0.0, 0.0, 0.0, wl.excitation]
        f0, amp = 2.87e9, configs.drive_amplitude(5e5)
    amp *= scale
    waves = []
    for k in range(points):
        w = Waveform(len(base), base=base)
        if k % 2:
            w.add(1, 1e-9, 5e-9 + 1e-10 * k, amp, 2 * np.pi * f0, 0.3)
            w.add(1, 9e-9, 2e-8, -amp, 2 * np.pi * f0, 0.1 * k)
        else:
            w.tone(1, amp, f0 + 1e6 * k)
        waves.append(w)
    sim = BatchSimulator(gens, 2, fine)
    dt = fine * H
    n_out = 600 // fine
    args = (waves, rho, 3e-10, 3e-10 + n_out * dt * (1 + 1e-9), dt)
    obs = None if read == "full" else obs
    print(f"{n} states x {points}, {read}", flush=True)
    got = sim.run(*args, obs=obs, read=read).cpu().numpy()
    assert sim.last_plan["series"] == orders, sim.last_plan
    want = sim.run(*args, obs=obs, read=read, taylor=17).cpu().numpy()
    assert got.shape == want.shape
    err = np.max(np.abs(got - want)) / np.max(np.abs(want))
    print(f"  {err:.1e}")
    assert err <= 1e-12


def test_models_beyond_the_kernels_rows_cost_no_matrices():
    _, weights, _ = quadratures.scheme(2)
    model = WideModel.build(*_model(193, 8), weights, H)
    assert model.plan(1e7, 1e-16) is None and len(model.mats) == 0


@pytest.mark.gpu
def test_full_states_whatever_the_count_of_readout_rows(gpu):
    """READ_FULL has no readout rows: the descriptor's count is not used."""
    wl = configs.odmr21(1, use_incoherent=True)
    sim = BatchSimulator(wl.generators, 2, 10)
    run = sim.prepare(wl.waveforms(), wl.rho0, 0.0, 1e-9, 2e-10, read="full")
    want = run.launch().cpu().numpy().copy()
    run.desc.n_obs = 40
    assert np.array_equal(run.launch().cpu().numpy(), want)


@pytest.mark.gpu
def test_launches_of_two_lds_sizes_at_once(gpu):
    """Two threads launch one kernel with different parts of LDS, each on its
    own stream, 300 times."""
    import threading

    import torch
    runs = []
    wl = configs.odmr21(1, use_incoherent=True)
    for scale, gens, rho, obs, base in (
            (6, wl.generators, wl.rho0, wl.obs,
             [1.0, 0.0, 0.0, 0.0, wl.excitation]),
            (10, np.stack(_model(112, 112)), np.ones((1, 112)) / 112,
             np.ones((1, 112)), [1.0, 0.0])):
        w = Waveform(len(base), base=base)
        amp = configs.drive_amplitude(5e5) if len(base) == 5 else 1e7
        w.tone(1, scale * amp, 2.87e9)
        sim = BatchSimulator(gens, 2, 3)
        run = sim.prepare([w], rho, 0.0, 3 * 6e-11 * (1 + 1e-9), 6e-11,
                          obs=obs)
        assert sim.last_plan["series"] == (2, 1)
        runs.append((run, run.launch().cpu().numpy().copy()))
    sizes = [run.desc.lds_columns for run, _ in runs]
    assert 0 < min(sizes) < max(sizes)
    failed = []

    def go(run, want):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(300):
                    run.launch()
                torch.cuda.current_stream().synchronize()
            if not np.array_equal(run.out.cpu().numpy(), want):
                failed.append(run)
        except Exception as error:      # the thread's own
            failed.append(error)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=go, args=r) for r in runs]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not failed, failed
