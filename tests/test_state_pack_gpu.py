"""State read-back around the size that one copy takes, in spin order after a
reorder, and after a step that raised the error flag."""
import numpy as np
import pytest

from dsim_amd import lib as D

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")


def _sub():
    return D.Substrate(np.zeros((0, 3), np.float32), np.zeros((0, 3), np.uint32),
                       np.zeros((0, 3), np.uint32), grid="aabb", dims=(8, 8, 8), lo=(-1.0,) * 3,
                       cell=(0.25,) * 3, device=True)


# 43690 spins: 4 + 6 n words are the whole of 2^18
@pytest.mark.parametrize("n", [1, 3, 257, 43690, 43691, 100003])
def test_state_round_trip(n):
    print(f"case state round trip {n}", flush=True)
    rng = np.random.default_rng(n)
    want = dict(pos=rng.uniform(-1, 1, (n, 3)).astype(np.float32),
                mag=rng.uniform(0, 1, n).astype(np.float32),
                phase=rng.normal(size=n).astype(np.float32),
                comp=rng.integers(0, 4, n).astype(np.uint8),
                fiber=rng.integers(0, 65536, n).astype(np.uint16))
    sub = _sub()
    sim = D.Simulation(sub, n, dt=0.005, std_dev=(0.01,) * 4, mode=D.MODE_PHYSICAL)
    sim.set_state(**want)
    got = sim.get_state()
    for k in want:
        np.testing.assert_array_equal(got[k], want[k])
    sim.close()
    sub.close()


@pytest.mark.parametrize("n", [1000, 60001])
def test_reordered_spins_come_back_in_spin_order(n):
    print(f"case state reordered {n}", flush=True)
    sub = _sub()
    out = []
    for sort in (0, 16):
        sim = D.Simulation(sub, n, dt=0.005, std_dev=(0.05,) * 4, mode=D.MODE_PHYSICAL,
                           boundary=D.BOUNDARY_PERIODIC, rng=D.RNG_PHILOX, seed=3,
                           sort_interval=sort)
        sim.init_uniform(1.0)
        sim.moment_reset()
        sim.integrate_moment(1.0, 48)
        out.append(sim.get_state())
        sim.close()
    for k in out[0]:
        np.testing.assert_array_equal(out[0][k], out[1][k])
    sub.close()
