"""Two readout rows through the Taylor queue kernel (GPU).

A wavefront runs several protocols one after another, some of no steps.
Each row of a two-row batch equals the batch that reads that row alone bit
for bit (the states and the sum over a row's components are the same
operations), and the first row the trapezoid of a sweep's every step at the
same degree to 1e-12 (the same states, added in another order: at most 3,000
additions of one rounding each, 3.3e-13).
"""

import numpy as np
import pytest

from superspinsim_amd import configs
from superspinsim_amd.protocols import ProtocolBatch, trapezoid_window
from superspinsim_amd.sweep import BatchSimulator

pytestmark = pytest.mark.gpu

H = 20e-12


@pytest.mark.parametrize("taylor,substeps,count,n_waves,wpb", [
    (17, None, 7, None, 1), (11, 1, 7, 2, 1), (12, 2, 9, 3, 2)])
def test_two_rows_equal_one_row(gpu, taylor, substeps, count, n_waves, wpb):
    wl = configs.pulsed7(count=count, seed=taylor, t_p_range=(2e-9, 4e-9),
                         tau_range=(5e-9, 2e-8), readout=10e-9)
    steps, read_from = wl.steps.copy(), wl.read_from.copy()
    steps[0], read_from[1] = 0, steps[1] + 5
    rng = np.random.default_rng(taylor)
    rho = np.abs(rng.standard_normal((count, wl.rho0.size))) * (wl.rho0 != 0)
    rows = np.concatenate([wl.obs, rng.standard_normal(wl.obs.shape)])

    def run(obs, noalloc=False):
        b = ProtocolBatch(wl.generators, 2).prepare(
            wl.waves, rho, H, steps, read_from, obs, taylor=taylor,
            substeps=substeps, n_waves=n_waves, waves_per_block=wpb)
        assert b.series is None
        print(f"{count} protocols, {obs.shape[0]} rows, degree {taylor}",
              flush=True)
        return (b.launch_noalloc() if noalloc else b.run()).cpu().numpy()

    got = run(rows)
    assert np.all(got[0] == 0) and np.all(got[1] == 0)
    assert np.all(got[2:] != 0)
    for k in range(2):
        assert np.array_equal(got[:, k], run(rows[k:k + 1])[:, 0])
    assert np.array_equal(run(rows, True), got)
    last = int(steps.max())
    assert last <= 3000
    trace = BatchSimulator(wl.generators, 2, 1).run(
        wl.waves, rho, 0.0, last * H * (1 + 1e-12), H, obs=rows[:1],
        taylor=taylor, substeps=substeps).cpu().numpy()[:, :, 0]
    want = trapezoid_window(
        np.concatenate([(rho @ rows[0])[:, None], trace], axis=1),
        read_from, steps, H)
    err = np.max(np.abs(got[:, 0] - want)) / np.max(np.abs(want))
    print(f"  {err:.1e}")
    assert err <= 1e-12
