"""Device blocks kept between simulation and waveform handles: several threads
creating, running and closing handles at once get the results that one thread
gets alone, and the blocks are given back with the last handle."""
import threading

import numpy as np
import pytest
import torch

from dsim_amd import lib as D
from dsim_amd import phase as PH

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")


def _work(sub, k, repeats):
    out = []
    for r in range(repeats):
        n = 3000 + 517 * ((k + r) % 4)
        sim = D.Simulation(sub, n, dt=0.005, std_dev=(0.02,) * 4, mode=D.MODE_PHYSICAL,
                           boundary=D.BOUNDARY_PERIODIC, rng=D.RNG_PHILOX, seed=k + 10 * r)
        sim.init_uniform(1.0)
        sim.label()
        sim.moment_reset()
        wf = PH.Waveforms(sim, PH.random_waveforms(40 + 100 * (k % 2), 64, seed=k), 0.37,
                          chunk_steps=32)
        wf.run(64)
        out += [wf.phase()[0], wf.signal(), sim.get_state()["pos"]]
        wf.close()
        sim.close()
    return out


def test_threads_share_the_pool_and_it_is_given_back():
    sub = D.Substrate(np.zeros((0, 3), np.float32), np.zeros((0, 3), np.uint32),
                      np.zeros((0, 3), np.uint32), grid="aabb", dims=(4, 4, 4), lo=(-1.0,) * 3,
                      cell=(0.5,) * 3, device=True)
    alone = [_work(sub, k, 3) for k in range(4)]
    before = torch.cuda.mem_get_info()[0]
    # a gigabyte through the pool
    sim = D.Simulation(sub, 200_000, dt=0.005, std_dev=(0.02,) * 4, mode=D.MODE_PHYSICAL,
                       boundary=D.BOUNDARY_PERIODIC, rng=D.RNG_PHILOX, seed=1)
    sim.init_uniform(1.0)
    sim.moment_reset()
    for _ in range(2):
        wf = PH.Waveforms(sim, PH.random_waveforms(512, 32, seed=3), 0.37, chunk_steps=32)
        wf.run(32)
        wf.close()
    kept = before - torch.cuda.mem_get_info()[0]
    got = [None] * 4
    ts = [threading.Thread(target=lambda k=k: got.__setitem__(k, _work(sub, k, 3)))
          for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    sim.close()
    for a, b in zip(alone, got):
        assert b is not None and len(a) == len(b)
        for x, y in zip(a, b):
            np.testing.assert_array_equal(x, y)
    assert kept > 300 << 20                  # the phases of 200,000 x 512 pairs
    assert before - torch.cuda.mem_get_info()[0] < 64 << 20
    sub.close()
