"""The flag of a step whose collision loop does not end, as each call that waits
reports it: once, and with the state valid afterwards."""
import os
import sys

import numpy as np
import pytest

from dsim_amd import lib as D

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [70, 50001])  # state in one copy, in several
@pytest.mark.parametrize("how", ["sync", "signal", "get_state"])
def test_endless_step_is_reported_once(how, n):
    print(f"case error flag through {how} spins {n}", flush=True)
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    from test_oracle_pins import _shared_diagonal_case
    env, pos, q = _shared_diagonal_case()
    P = np.random.default_rng(3).uniform(-0.9, 0.9, (n, 3)).astype(np.float32)
    Q = np.zeros((1, n, 4), np.float32)
    Q[..., 3] = 0.5
    P[37], Q[0, 37] = pos[0], q[0, 0]
    sub = D.Substrate(env["vertices"], env["triangles"], env["tri_info"])
    sim = D.Simulation(sub, n, dt=0.005, std_dev=env["std_dev"], t2=env["t2"], mode=D.MODE_REFERENCE)
    sim.set_state(pos=P, comp=np.zeros(n, np.uint8), fiber=np.full(n, D.NO_FIBER, np.uint16))
    sim.integrate_injected(np.zeros(3, np.float32), 0.0, Q)
    with pytest.raises(D.DsimError) as e:
        getattr(sim, how)()
    assert e.value.code == -5
    s = sim.get_state()
    other = np.arange(n) != 37
    np.testing.assert_array_equal(s["pos"][other], P[other])  # they did not move
    assert sim.signal()[0] > 0.0
    sim.sync()
    sim.close()
    sub.close()
