"""The labeller's pass over all triangles (reference semantics, and re-casts):
triangle counts around its tiles of 256, spin counts around its blocks, both
triangle tests, all membrane types, against the oracle's labels."""
import os
import sys

import numpy as np
import pytest

import oracle as O
from dsim_amd import lib as D

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from test_walk_soup_gpu import _soup  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tris,n", [(1, 1), (255, 255), (256, 257), (257, 1000), (300, 4097)])
def test_labels_match_oracle(tris, n):
    print(f"case label pass triangles {tris} spins {n}", flush=True)
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    V, T, I = _soup(260, 17)
    T, I = T[:tris], I[:tris].copy()
    I[:, 0] %= 5
    I[:, 1] = np.arange(tris) % 3
    pos = np.random.default_rng(n).uniform(-0.95, 0.95, (n, 3)).astype(np.float32)
    w = O.World(V, T, I, std_dev=(0.01,) * 4, t2=(80.0,) * 4, dt=0.005, n_cubes=10)
    comp, fib, tries, amb = w.find_spins(pos, 1.3, 1.3, 1.3, max_tries=0)
    sub = D.Substrate(V, T, I, device=True, n_cubes=10)
    sim = D.Simulation(sub, n, dt=0.005, std_dev=(0.01,) * 4, mode=D.MODE_REFERENCE, rng=D.RNG_MWC)
    sim.set_state(pos=pos)
    # a ray that leaves two fibres of a membrane type open keeps either's label
    assert sim.label(1.3, 1.3, 1.3, max_tries=0) == amb
    s, clear = sim.get_state(), tries == 0
    np.testing.assert_array_equal(s["comp"][clear], comp[clear])
    np.testing.assert_array_equal(s["fiber"][clear], fib[clear])
    assert n == 1 or clear.sum() > n // 2
    sim.close()
    sub.close()
