"""Labels where many triangles reach past the grid's far face over many rows:
they stand in one list that the rows share, and labelling takes no memory for an
entry per row and triangle."""
import os
import sys

import numpy as np
import pytest
import torch

from dsim_amd import lib as D

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from test_label_rows_gpu import _mesh  # noqa: E402

pytestmark = pytest.mark.gpu


def _with_walls(V, T, I, axis, face, seed):
    """Adds triangles across the rays around the grid's face, each over most of
    the grid's rows."""
    rng = np.random.default_rng(seed)
    W = rng.uniform(-1.2, 1.2, (220, 3, 3))
    W[:, :, axis] = rng.uniform(face - 0.02, face + 0.3, (220, 1)) + rng.uniform(0, 0.03, (220, 3))
    J = np.stack([np.arange(220) % 40, np.arange(220) % 3, len(V) + 3 * np.arange(220)], 1)
    U = len(V) + np.arange(660).reshape(220, 3)
    return (np.concatenate([V, W.reshape(-1, 3)]).astype(np.float32),
            np.concatenate([T, U]).astype(np.uint32), np.concatenate([I, J]).astype(np.uint32))


# the last: one cell, whose row lists every triangle
@pytest.mark.parametrize("axis,grid,dims,n", [
    (0, "aabb", (4, 600, 600), 3001), (2, "aabb", (500, 700, 3), 40001),
    (1, "tribox", (500, 3, 500), 2049), (0, "aabb", (1, 1, 1), 65)])
def test_triangles_past_the_grid(axis, grid, dims, n):
    print(f"case past the grid axis {axis} {grid} {dims} spins {n}", flush=True)
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    V, T, I = _with_walls(*_mesh(axis, 9, 60), axis, -0.1, n)
    pos = np.random.default_rng(n).uniform(-0.95, 0.95, (n, 3)).astype(np.float32)
    pos[:, axis] *= 0.6
    lo, hi = np.array([-1.0, -0.9, -0.8]), np.array([0.9, 0.95, 0.98])
    hi[axis] = -0.1  # most of the mesh reaches beyond it
    sub = D.Substrate(V, T, I, device=True, grid=grid, dims=dims, lo=tuple(lo),
                      cell=tuple((hi - lo) / dims), eps=1e-5, clearance_rings=1)
    assert sub.label_axis() == axis
    assert sub.nbytes() < 256 << 20
    out = []
    for s in (D.Substrate(V, T, I, device=True, n_cubes=10), sub):
        sim = D.Simulation(s, n, dt=0.005, std_dev=(0.01,) * 4, mode=D.MODE_PHYSICAL)
        sim.set_state(pos=pos)
        before = torch.cuda.mem_get_info()[0]
        amb = sim.label(1.3, 1.3, 1.3, max_tries=2)
        # its blocks are kept: what the call took is still taken
        assert before - torch.cuda.mem_get_info()[0] < 64 << 20
        st = sim.get_state()
        out.append((amb, st["comp"], st["fiber"]))
        sim.close()
        s.close()
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1:], out[1][1:]):
        np.testing.assert_array_equal(a, b)
    assert n < 100 or (out[0][1] > 0).sum() > n // 20
