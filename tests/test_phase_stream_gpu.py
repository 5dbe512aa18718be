"""A walk started right after its waveforms are created (or given another
trajectory buffer) records what a walk started on an idle device records: the
clearing of the phases and of the trajectory buffer is ordered before it."""
import numpy as np
import pytest

from dsim_amd import lib as D
from dsim_amd import phase as PH
from dsim_amd import substrate as S

pytestmark = pytest.mark.gpu

GAMMA = 42576.0


@pytest.mark.parametrize("buffer", [64, 512])
def test_walk_right_after_create(buffer):
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    cfg = S.SMALL
    e = S.build(cfg, cell_um=0.5, axons=S.pack(cfg))
    g = e["grid"]
    sub = D.Substrate(e["vertices"], e["triangles"], e["tri_info"], grid="aabb", dims=g["dims"],
                      lo=g["lo"], cell=g["cell"], eps=g["eps"])
    # 250,000 spins: buffers of 0.2-1.5 GB, whose clearing takes as long as
    # many steps of the walk
    n, n_wave, steps, chunk = 250_000, 128, 512, 64
    pc = np.float32(2 * np.pi * GAMMA * cfg.dt)
    w = PH.random_waveforms(n_wave, steps, seed=3) * np.float32(1e-9 * e["space_scale"])
    out = []
    for idle in (True, False):
        print(f"waveforms: {n} spins, buffer {buffer}, idle {idle}", flush=True)
        sim = D.Simulation(sub, n, dt=cfg.dt, std_dev=e["std_dev"], mode=D.MODE_PHYSICAL,
                           boundary=D.BOUNDARY_PERIODIC, seed=8)
        sim.init_uniform(1.0)
        sim.moment_reset()
        wf = PH.Waveforms(sim, w, pc, chunk_steps=chunk, buffer_steps=buffer)
        if idle:
            D.check(D.lib().dsim_thread_sync())
        wf.run(steps)
        out.append(wf.phase())
        wf.close()
        sim.close()
    sub.close()
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
    assert np.abs(out[0][0]).max() > 1e-3
