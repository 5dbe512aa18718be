"""Trajectories and phases of waveform runs do not depend on how the steps are
split into launches: launch lengths and reorder intervals that are no multiple
of the four steps that a trajectory tile's chunks of rows take together."""
import numpy as np
import pytest

from dsim_amd import lib as D
from dsim_amd import phase as PH

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 129, 5000])
@pytest.mark.parametrize("rng", [D.RNG_PHILOX, D.RNG_MWC])
def test_launch_lengths_leave_the_trajectory(n, rng):
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    sub = D.Substrate(np.zeros((0, 3), np.float32), np.zeros((0, 3), np.uint32),
                      np.zeros((0, 3), np.uint32), grid="aabb", dims=(4, 4, 4), lo=(-1.0,) * 3,
                      cell=(0.5,) * 3, device=True)
    g = PH.random_waveforms(3, 96, seed=n)
    want = None
    for spl, sort in [(0, 0), (1, 0), (3, 0), (7, 0), (30, 0), (0, 5), (7, 10), (2, 3)]:
        print(f"case launches of {spl}, reorders after {sort}, spins {n}, rng {rng}", flush=True)
        sim = D.Simulation(sub, n, dt=0.005, std_dev=(0.01,) * 4, mode=D.MODE_PHYSICAL,
                           boundary=D.BOUNDARY_PERIODIC, rng=rng, seed=4, sort_interval=sort,
                           steps_per_launch=spl)
        sim.init_uniform(1.0)
        sim.moment_reset()
        wf = PH.Waveforms(sim, g, 0.37, chunk_steps=32, buffer_steps=64)
        out = (wf.run(96, trajectory=True),) + wf.phase()
        wf.close()
        sim.close()
        if want is None:
            want = out
            assert np.isfinite(out[0]).all() and np.abs(out[0]).min(axis=(1, 2)).max() > 0
        for a, b in zip(out, want):
            np.testing.assert_array_equal(a, b)
    sub.close()
