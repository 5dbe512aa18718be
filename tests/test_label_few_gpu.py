"""Labelling a few spins on an AABB grid of many cells reads row lists that the
substrate holds: the call builds none of its own, whose making would take longer
than walking the rows."""
import numpy as np
import pytest
import torch

from dsim_amd import lib as D
from dsim_amd import substrate as S

pytestmark = pytest.mark.gpu


def test_few_spins_on_a_large_aabb_grid():
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    cfg = S.SMALL
    e = S.build(cfg, cell_um=0.5, axons=S.pack(cfg))
    print("case few spins, 400^3 cells", flush=True)
    out = []
    for dims in ((400, 400, 400), (50, 50, 50)):
        sub = D.Substrate(e["vertices"], e["triangles"], e["tri_info"], device=True, grid="aabb",
                          dims=dims, lo=(-1.05,) * 3, cell=(2.1 / dims[0],) * 3, eps=1e-5,
                          clearance_rings=1)
        sim = D.Simulation(sub, 1000, dt=cfg.dt, std_dev=e["std_dev"], mode=D.MODE_PHYSICAL,
                           boundary=D.BOUNDARY_PERIODIC, seed=3)
        sim.init_uniform(1.0)
        sim.sync()
        before = torch.cuda.mem_get_info()[0]
        amb = sim.label(*(e["xmax"],) * 3)
        # blocks of the call stay allocated while a simulation is alive
        assert before - torch.cuda.mem_get_info()[0] < 16 << 20
        st = sim.get_state()
        out.append((amb, st["comp"], st["fiber"]))
        sim.close()
        sub.close()
    assert out[0][0] == out[1][0] == 0
    np.testing.assert_array_equal(out[0][1], out[1][1])
    np.testing.assert_array_equal(out[0][2], out[1][2])
    assert (out[0][1] > 0).sum() > 100
