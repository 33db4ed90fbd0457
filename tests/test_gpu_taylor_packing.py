"""Several instances of a small model per wavefront on the Taylor path (GPU):
runs that name a Taylor degree, and time chunks of a model with two driven
generators.  A row of a block sums the single-instance row's terms plus
exact zeros, only in another order: 1e-13 relative, as for the packed runs of
the series; chunks chain their propagators, a few ulp each: 1e-12."""

import numpy as np
import pytest

from superspinsim_amd import configs

pytestmark = pytest.mark.gpu


def _run(wl, waves, n_out, pack, read, taylor=11):
    sim = wl.simulator()
    sim.pack = pack
    out = sim.run(waves, wl.rho0, 0.0, n_out * wl.time_step * (1 + 1e-12),
                  wl.time_step, obs=None if read == "full" else wl.obs,
                  read=read, taylor=taylor)
    assert "series" not in sim.last_plan
    return out.cpu().numpy(), sim.last_plan["packed"]


@pytest.mark.parametrize("model,points,n_out,pack,read", [
    ("nv7c", 5, 6, 2, "obs"), ("nv7c", 5, 6, 2, "integral"),
    ("nv7c", 5, 6, 2, "full"), ("nv3", 9, 20, 7, "full"),
    ("nv7c", 4096, 5, True, "obs")])
def test_packed_equals_unpacked(gpu, model, points, n_out, pack, read):
    wl = configs.odmr3(points) if model == "nv3" else \
        configs.odmr7(points, use_incoherent=True)
    wl.frequencies = np.linspace(2.80e9, 2.94e9, points)
    waves = wl.waveforms()
    packed, k = _run(wl, waves, n_out, pack, read)
    plain, one = _run(wl, waves, n_out, False, read)
    assert (k, one) == (2 if pack is True else pack, 1)
    assert packed.shape == plain.shape and packed.shape[0] == points
    d = np.max(np.abs(packed - plain)) / np.max(np.abs(plain))
    print(f"{model} x {points} {read}: {d:.1e}", flush=True)
    assert d <= 1e-13


@pytest.mark.parametrize("read,chunks", [("obs", 7), ("full", 3)])
def test_chunks_of_two_drives_equal_run(gpu, read, chunks):
    wl = configs.odmr3(1)
    waves = []
    for k in range(3):
        w = wl.waveform(2.8e9 + 5e7 * k)
        w.tone(2, 0.5 * wl.b1, 2.75e9)
        waves.append(w)
    sim = wl.simulator()
    args = (waves, wl.rho0, 2e-9, 2e-9 + 50 * wl.time_step * (1 + 1e-9),
            wl.time_step)
    obs = None if read == "full" else wl.obs
    want = sim.run(*args, obs=obs, read=read).cpu().numpy()
    got = sim.run_chunked(*args, obs=obs, read=read,
                          chunks=chunks).cpu().numpy()
    assert "series" not in sim.last_plan
    assert sim.last_plan["chunk_pack"] > 1
    err = np.max(np.abs(got - want)) / np.max(np.abs(want))
    print(f"{read}: {err:.1e}", flush=True)
    assert err <= 1e-12
