"""A waveform handle in blocks that others left: the first product starts from
zero and the padded part of the trajectory is never cleared, so phases,
compensations and signals have to be those of clean memory whatever the blocks
hold, beside odd spin counts whose last pair is half padding."""
import numpy as np
import pytest

from dsim_amd import lib as D
from dsim_amd import phase as PH

pytestmark = pytest.mark.gpu


def _handle(sub, n, grads, seed=6, buffer=None):
    sim = D.Simulation(sub, n, dt=0.005, std_dev=(0.01,) * 4, mode=D.MODE_PHYSICAL,
                       boundary=D.BOUNDARY_PERIODIC, rng=D.RNG_PHILOX, seed=seed)
    sim.init_uniform(1.0)
    sim.moment_reset()
    return sim, PH.Waveforms(sim, grads, 0.37, chunk_steps=32, buffer_steps=buffer)


@pytest.mark.parametrize("n,n_wave,buffer", [(1, 1, 32), (129, 130, 32), (4097, 257, 64),
                                             (20001, 128, 64)])
def test_blocks_of_other_handles(n, n_wave, buffer):
    print(f"case dirty blocks spins {n} waveforms {n_wave} buffer {buffer}", flush=True)
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    D.trim_memory()
    sub = D.Substrate(np.zeros((0, 3), np.float32), np.zeros((0, 3), np.uint32),
                      np.zeros((0, 3), np.uint32), grid="aabb", dims=(4, 4, 4), lo=(-1.0,) * 3,
                      cell=(0.5,) * 3, device=True)
    # the blocks wait for the next handle while a simulation is alive
    keep = D.Simulation(sub, 1, dt=0.005, std_dev=(0.01,) * 4, mode=D.MODE_PHYSICAL)
    g = PH.random_waveforms(n_wave, 128, seed=n)
    out = []
    for dirty in (False, True):
        if dirty:
            D.trim_memory()
            # handles of the same sizes, phases and trajectories NaN and infinite
            bad = np.full_like(g, np.inf)
            bad[:, ::2] = np.nan
            for k in range(2):
                sim, wf = _handle(sub, n + (n % 128 != 0) * k, bad, seed=9, buffer=buffer)
                wf.run(128)
                assert not np.isfinite(wf.phase()[0]).any()
                wf.close()
                st = sim.get_state()
                sim.set_state(pos=np.full_like(st["pos"], np.nan))
                sim.moment_reset()
                wf = PH.Waveforms(sim, g, 0.37, chunk_steps=32, buffer_steps=buffer)
                wf.run(128)
                wf.close()
                sim.close()
        sim, wf = _handle(sub, n, g, buffer=buffer)
        first = wf.signal()
        wf.run(64)
        half = wf.phase()
        wf.run(64)
        out.append((first, *half, *wf.phase(), wf.signal()))
        wf.close()
        sim.close()
    keep.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, b)
    sub.close()
