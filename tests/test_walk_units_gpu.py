"""The physical-mode walk on meshes and grids in other units than the normalised
ones: steps aimed at the edges of triangles, where the searches' bounds may
round, hit what the oracle's do, bit for bit."""
import os
import sys

import numpy as np
import pytest

import oracle as O
from dsim_amd import lib as D

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from test_walk_soup_gpu import GRIDS, T2, DT, _soup  # noqa: E402

pytestmark = pytest.mark.gpu


def _at_edges(V, T, n, unit, rng):
    """Starts and steps of segments through points of the triangles' longest
    edges, and of their vertices."""
    tri = V[T[rng.integers(len(T), size=n)]].astype(np.float64)
    e = tri[:, [1, 2, 2]] - tri[:, [0, 0, 1]]
    k = (e ** 2).sum(-1).argmax(1)
    a = tri[np.arange(n), np.array([0, 0, 1])[k]]
    t = np.where(rng.uniform(size=n) < 0.8, rng.uniform(size=n), 0.0)[:, None]
    at = a + t * e[np.arange(n), k]
    d = rng.normal(size=(n, 3))
    d *= (unit * rng.uniform(0.01, 0.1, n) / np.linalg.norm(d, axis=1))[:, None]
    s = rng.uniform(0.05, 0.95, (n, 1))
    return (at - s * d).astype(np.float32), d.astype(np.float32)


@pytest.mark.parametrize("unit,shift", [(1.0, 0.0), (256.0, 0.0), (4096.0, 0.0), (1.0, 300.0)])
@pytest.mark.parametrize("grid", ["aabb-3d", "aabb-plane", "tribox-3d"])
def test_edges_are_hit_in_any_units(grid, unit, shift):
    print(f"case units {grid} unit {unit} shift {shift}", flush=True)
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    V, T, I = _soup(240, 3)
    # one triangle a wall, none degenerate: a step along an edge that two share
    # may hit them in turn without end
    keep = np.unique(T.min(1), return_index=True)[1]
    a, b, c = (V[T[keep, k]].astype(np.float64) for k in range(3))
    keep = keep[np.linalg.norm(np.cross(b - a, c - a), axis=1) > 1e-6]
    T, I = T[keep], I[keep]
    V = (V * np.float32(unit) + np.float32(shift)).astype(np.float32)
    pos, step = _at_edges(V, T, 500_000, unit, np.random.default_rng(7))
    # within the grid, outside which an exact-membership grid lists nothing
    inside = (np.abs(pos - np.float32(shift)).max(1) < 1.15 * unit)
    pos, step = pos[inside], step[inside]
    n = len(pos)
    q = np.zeros((1, n, 4), np.float32)
    q[0, :, :3] = step
    q[0, :, 3] = 0.5

    def put(g):
        lo = tuple(float(np.float32(v * unit + shift)) for v in g["lo"])
        cell = tuple(float(np.float32(v * unit)) for v in g["cell"])
        return dict(g, lo=lo, cell=cell, eps=float(np.float32(max(1e-5 * unit, 1e-6 * shift))))

    box = ((-3.0 * unit + shift,) * 3, (3.0 * unit + shift,) * 3)
    w = O.World(V, T, I, std_dev=(1.0,) * 4, t2=T2, dt=DT, permeability=1.0, test=1, traversal=1,
                transitions=1, boundary=1, voxel_lo=box[0], voxel_hi=box[1],
                **put(GRIDS["aabb-3d" if grid == "tribox-3d" else grid]))
    st = O.State(pos, comp=np.zeros(n, np.uint8), fiber=np.full(n, D.NO_FIBER, np.uint16), moment=True)
    to = O.integrate(w, st, 1, rng=O.RNG_INJECT, inject=q, weight=1.0, trace=True)
    ends = to[0, :, 2] < 4096  # not a step that hits two triangles' common points without end
    pos, q, to, want, n = pos[ends], q[:, ends], to[:, ends], st.pos[ends], int(ends.sum())
    assert n > 300_000
    sub = D.Substrate(V, T, I, device=True, **put(GRIDS[grid]))
    sim = D.Simulation(sub, n, dt=DT, std_dev=(1.0,) * 4, t2=T2, permeability=1.0, mode=D.MODE_PHYSICAL,
                       boundary=D.BOUNDARY_PERIODIC, seed=5, voxel=box)
    sim.set_state(pos=pos, comp=np.zeros(n, np.uint8))
    sim.moment_reset()
    tg = sim.integrate_moment_injected(1.0, q, trace=True)
    np.testing.assert_array_equal(tg[..., [0, 1, 2, 4]], to[..., [0, 1, 2, 4]])
    np.testing.assert_array_equal(sim.get_state()["pos"], want)
    assert (to[..., 2] > 0).sum() > n // 4
    sim.close()
    sub.close()
