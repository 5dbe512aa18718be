"""The grid-row labeller against the pass over all triangles, on triangle soups
(every ray's first result is kept, ambiguous or not): each ray axis, planar and
exact-membership grids whose faces cut through the mesh, spins outside the grid
box, spin counts that leave blocks partly filled, and spins ordered by row."""
import os
import sys

import numpy as np
import pytest

from dsim_amd import lib as D

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from test_walk_soup_gpu import _soup  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")


def _mesh(axis, seed, tris=160):
    V, T, I = _soup(tris, seed)
    V = V.copy()
    if axis:  # the walls (along z) along x
        V = V[:, [2, 1, 0]]
    V[:, axis] *= 0.5  # least extent along the ray axis
    I = I.copy()
    I[:, 1] = np.arange(len(T)) % 3
    return np.ascontiguousarray(V, np.float32), T, I


@pytest.mark.parametrize("axis,grid,dims,n", [
    (0, "aabb", (24, 20, 1), 1),
    (0, "aabb", (24, 20, 16), 5001),
    (1, "aabb", (7, 30, 9), 4097),
    (2, "aabb", (11, 8, 21), 31),
    (0, "tribox", (24, 20, 16), 5001),
    (1, "tribox", (12, 9, 30), 999),
    (2, "tribox", (10, 10, 10), 33),
    (0, "aabb", (4, 512, 512), 32768),     # ordered by row: rows past the L2's size
    (2, "aabb", (300, 300, 4), 40001),
    (0, "tribox", (58, 760, 764), 20001),  # lists too large to keep, made by the call
])
def test_rows_match_the_pass_over_all_triangles(axis, grid, dims, n):
    print(f"case label rows axis {axis} {grid} {dims} spins {n}", flush=True)
    V, T, I = _mesh(axis, 5, 12 if dims[1] > 700 else 160)
    pos = np.random.default_rng(n).uniform(-0.95, 0.95, (n, 3)).astype(np.float32)
    pos[:, axis] *= 0.6
    lo, hi = np.array([-1.0, -0.9, -0.8]), np.array([0.7, 0.8, 0.9])
    hi[axis] = 0.25  # triangles beyond it
    sub = D.Substrate(V, T, I, device=True, grid=grid, dims=dims, lo=tuple(lo),
                      cell=tuple((hi - lo) / dims), eps=1e-5, clearance_rings=1)
    assert sub.label_axis() == axis
    out = []
    for s in (D.Substrate(V, T, I, device=True, n_cubes=10), sub):
        sim = D.Simulation(s, n, dt=0.005, std_dev=(0.01,) * 4, mode=D.MODE_PHYSICAL)
        got = []
        for max_tries in (0, 2):
            sim.set_state(pos=pos)
            amb = sim.label(1.3, 1.3, 1.3, max_tries=max_tries)
            st = sim.get_state()
            got.append((amb, st["comp"], st["fiber"]))
        out.append(got)
        sim.close()
        s.close()
    for a, b in zip(*out):
        assert a[0] == b[0]
        np.testing.assert_array_equal(a[1], b[1])
        np.testing.assert_array_equal(a[2], b[2])
    assert n < 100 or (out[0][0][1] > 0).sum() > n // 20
