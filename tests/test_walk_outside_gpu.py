"""The physical-mode walk past a grid smaller than its mesh.  An exact-membership
grid lists a triangle in the cells that it meets and nowhere for its part outside
the box; a step that leaves the box is tested against all the lists from its start's
cell to its end's (the nearest one in the grid), whatever the clearance there."""
import numpy as np
import pytest

import oracle as O
from dsim_amd import lib as D

pytestmark = pytest.mark.gpu

T2, DT = (80.0, 70.0, 7.5, 70.0), 0.005
LO, CELL, DIMS = -1.0, np.float32(0.125), (16, 16, 1)
TRI = np.array([[-0.31, -0.22, -0.42], [0.47, 0.13, -1.72], [-0.12, 0.61, -1.65]])


def _steps(n, rng):
    """Steps from inside the grid through the triangle's part below its floor,
    whose box of cells holds one that the triangle meets inside."""
    pos = rng.uniform((-0.99,) * 3, (0.99, 0.99, -0.2), (n, 3)).astype(np.float32)
    inside, at = rng.dirichlet((1.0, 1.0, 1.0), (2, n)) @ TRI
    step = ((at - pos) * rng.uniform(1.05, 1.5, (n, 1))).astype(np.float32)
    ends = np.sort(np.stack([pos, pos + step])[..., :2], 0)
    low, high = np.clip(np.floor((ends - LO) / CELL), 0, DIMS[0] - 1)
    cells = np.floor((inside[None, :, :2] + np.array([[[1e-4]], [[-1e-4]]]) - LO) / CELL)
    ok = (inside[:, 2] > -0.99) & (at[:, 2] < -1.01)
    ok &= (cells >= low).all((0, 2)) & (cells <= high).all((0, 2))
    return pos[ok], step[ok]


@pytest.mark.parametrize("grid", ["tribox", "aabb"])
def test_steps_that_leave_the_grid_hit_past_it(grid):
    print(f"case past the grid {grid}", flush=True)
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    V, T = TRI.astype(np.float32), np.array([[0, 1, 2]], np.uint32)
    I = np.array([[3, 0, 0]], np.uint32)
    pos, step = _steps(800_000, np.random.default_rng(8))
    n = len(pos)
    assert n > 10_000
    q = np.zeros((1, n, 4), np.float32)
    q[0, :, :3] = step
    q[0, :, 3] = 0.5
    w = O.World(V, T, I, std_dev=(1.0,) * 4, t2=T2, dt=DT, permeability=1.0, test=1, traversal=1,
                transitions=1, boundary=0, grid="aabb", dims=(1, 1, 1), lo=(-2.0,) * 3,
                cell=(4.0,) * 3, eps=1e-5)
    st = O.State(pos, comp=np.zeros(n, np.uint8), fiber=np.full(n, D.NO_FIBER, np.uint16), moment=True)
    to = O.integrate(w, st, 1, rng=O.RNG_INJECT, inject=q, weight=1.0, trace=True)
    sub = D.Substrate(V, T, I, device=True, grid=grid, dims=DIMS, lo=(LO,) * 3,
                      cell=(float(CELL), float(CELL), 2.0), eps=1e-5)
    sim = D.Simulation(sub, n, dt=DT, std_dev=(1.0,) * 4, t2=T2, permeability=1.0, mode=D.MODE_PHYSICAL,
                       boundary=D.BOUNDARY_CLAMP, seed=5)
    sim.set_state(pos=pos, comp=np.zeros(n, np.uint8))
    sim.moment_reset()
    tg = sim.integrate_moment_injected(1.0, q, trace=True)
    assert (to[..., 2] > 0).sum() > n // 2
    np.testing.assert_array_equal(tg[..., [0, 1, 2, 4]], to[..., [0, 1, 2, 4]])
    np.testing.assert_array_equal(sim.get_state()["pos"], st.pos)
    sim.close()
    sub.close()
