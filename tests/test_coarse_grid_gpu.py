"""Grids of few cells with many triangles each, whose lists a block builds
together: the walk against the oracle bit for bit, the row labels against the
pass over all triangles, list lengths around the 64 that a thread takes alone
and the 256 of a block, and the time of a build."""
import os
import sys
import time

import numpy as np
import pytest

import oracle as O
from dsim_amd import lib as D

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from test_walk_soup_gpu import _soup  # noqa: E402

pytestmark = pytest.mark.gpu

STD, T2, DT = (0.05, 0.04, 0.03, 0.05), (80.0, 70.0, 7.5, 70.0), 0.005


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")


@pytest.mark.parametrize("grid", ["aabb", "tribox"])
@pytest.mark.parametrize("dims,tris", [((1, 1, 1), 64), ((1, 1, 1), 65), ((1, 1, 1), 256),
                                       ((1, 1, 1), 257), ((2, 1, 1), 700), ((2, 3, 2), 900),
                                       ((5, 4, 3), 900)])
def test_walk_and_labels(dims, tris, grid):
    print(f"case coarse grid {grid} {dims} triangles {tris}", flush=True)
    V, T, I = _soup(640, 21)
    T, I = T[:tris], I[:tris].copy()
    I[:, 1] = np.arange(tris) % 3
    lo, cell = (-1.3,) * 3, tuple(2.6 / d for d in dims)
    n, iters = 600, 12
    rng = np.random.default_rng(tris)
    pos = rng.uniform(-0.95, 0.95, (n, 3)).astype(np.float32)
    comp = rng.integers(0, 3, n).astype(np.uint8)
    q = rng.normal(size=(iters, n, 4)).astype(np.float32)
    q[..., 3] = rng.uniform(0, 1, (iters, n))
    w = O.World(V, T, I, std_dev=STD, t2=T2, dt=DT, permeability=0.3, test=1, traversal=1,
                transitions=1, boundary=0, grid="aabb", dims=dims, lo=lo, cell=cell, eps=1e-5)
    st = O.State(pos, comp=comp, fiber=np.full(n, D.NO_FIBER, np.uint16), moment=True)
    to = O.integrate(w, st, iters, rng=O.RNG_INJECT, inject=q, weight=1.0, trace=True)
    sub = D.Substrate(V, T, I, device=True, grid=grid, dims=dims, lo=lo, cell=cell, eps=1e-5)
    sim = D.Simulation(sub, n, dt=DT, std_dev=STD, t2=T2, permeability=0.3, mode=D.MODE_PHYSICAL)
    sim.set_state(pos=pos, comp=comp)
    sim.moment_reset()
    tg = sim.integrate_moment_injected(1.0, q, trace=True)
    np.testing.assert_array_equal(tg[..., [0, 1, 2, 4]], to[..., [0, 1, 2, 4]])
    np.testing.assert_array_equal(sim.get_state()["pos"], st.pos)
    sim.close()
    out = []
    for s in (D.Substrate(V, T, I, device=True, n_cubes=10), sub):
        sim = D.Simulation(s, n, dt=DT, std_dev=STD, mode=D.MODE_PHYSICAL)
        sim.set_state(pos=pos)
        amb = sim.label(1.3, 1.3, 1.3, max_tries=2)
        g = sim.get_state()
        out.append((amb, g["comp"], g["fiber"]))
        sim.close()
        s.close()
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1:], out[1][1:]):
        np.testing.assert_array_equal(a, b)


def test_build_of_one_full_cell_is_not_serial():
    n = 60_000
    rng = np.random.default_rng(5)
    V = (rng.uniform(-1, 1, (n, 1, 3)) + rng.uniform(-0.05, 0.05, (n, 3, 3))).reshape(-1, 3)
    T = np.arange(3 * n).reshape(n, 3)
    I = np.stack([np.arange(n) % 50, np.zeros(n, int), T[:, 0]], 1)
    best = 1e9
    for _ in range(2):
        print(f"case one cell, {n} triangles", flush=True)
        t = time.perf_counter()
        sub = D.Substrate(V, T, I, device=True, grid="aabb", dims=(1, 1, 1), lo=(-1.3,) * 3,
                          cell=(2.6,) * 3, eps=1e-5)
        D.check(D.lib().dsim_thread_sync())
        best = min(best, time.perf_counter() - t)
        sub.close()
    print(f"build {best * 1e3:.1f} ms", flush=True)
    assert best < 0.05  # a few ms; a thread over the list takes tens and more
