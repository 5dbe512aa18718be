"""The waveform handle's device-side preparation and read-back: phases before
any run are zero, a waveform's phases do not depend on the others beside it
(tiles of either width, padded or not), and phases come back whole where the
rows pass the read-back's staging buffer, for odd spin counts."""
import numpy as np
import pytest

from dsim_amd import lib as D
from dsim_amd import phase as PH

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")


def _run(n, grads, runs, chunk):
    sub = D.Substrate(np.zeros((0, 3), np.float32), np.zeros((0, 3), np.uint32),
                      np.zeros((0, 3), np.uint32), grid="aabb", dims=(4, 4, 4), lo=(-1.0,) * 3,
                      cell=(0.5,) * 3, device=True)
    sim = D.Simulation(sub, n, dt=0.005, std_dev=(0.01,) * 4, mode=D.MODE_PHYSICAL,
                       boundary=D.BOUNDARY_PERIODIC, rng=D.RNG_PHILOX, seed=4)
    sim.init_uniform(1.0)
    sim.moment_reset()
    wf = PH.Waveforms(sim, grads, 0.37, chunk_steps=chunk)
    first = wf.signal(), wf.phase()
    for steps in runs:
        wf.run(steps)
    out = wf.phase() + (wf.signal(),)
    wf.close()
    sim.close()
    sub.close()
    return first, out


# 1003 waveforms: 20001 rows of 4012 bytes pass the 64 MB staging buffer
@pytest.mark.parametrize("n,n_wave,steps,chunk", [(20001, 1003, 32, 32), (1, 1, 96, 64),
                                                  (129, 385, 64, 32)])
def test_phases_are_whole_and_independent(n, n_wave, steps, chunk):
    print(f"case phase blocks spins {n} waveforms {n_wave} steps {steps}", flush=True)
    g = PH.random_waveforms(n_wave, steps, seed=n)
    g[:, -1] = np.float32(1e-39)                      # a subnormal product
    (s0, (p0, c0)), (p, c, s) = _run(n, g, [32] * (steps // 32), chunk)
    assert not p0.any() and not c0.any()
    assert (s0[:, 0] <= 1.0 + 1e-12).all() and (s0[:, 0] > 0.0).all()
    assert np.isfinite(p).all() and (n_wave == 1 or np.abs(p).max() > 0)
    for w in sorted({0, n_wave // 2, n_wave - 1}):
        _, (q, d, t) = _run(n, np.ascontiguousarray(g[:, w:w + 1]), [32] * (steps // 32), chunk)
        np.testing.assert_array_equal(p[:, w], q[:, 0])
        np.testing.assert_array_equal(c[:, w], d[:, 0])
        np.testing.assert_array_equal(s[w], t[0])
