"""The reference-mode steps (k_ref_walk) where their search can go wrong, bit
for bit against the oracle on injected steps: boxes of more cells than a
search round lists, cells of many triangles and of none, degenerate triangles,
lists read through cell_tri (grids other than the reference's), spin counts
that leave waves partly filled; and a step whose collision loop does not end,
among spins whose steps do."""
import os
import sys

import numpy as np
import pytest

import oracle as O
from dsim_amd import lib as D

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from test_walk_soup_gpu import _soup  # noqa: E402

pytestmark = pytest.mark.gpu

T2, DT = (80.0, 70.0, 7.5, 70.0), 0.005
AABB = dict(grid="aabb", dims=(24, 20, 16), lo=(-1.3,) * 3, cell=(2.6 / 24, 2.6 / 20, 2.6 / 16),
            eps=1e-5)


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")


def soup_case(n, iters, std, n_cubes, seed):
    V, T, I = _soup(160, seed)
    rng = np.random.default_rng(seed + 1)
    pos = rng.uniform(-0.9, 0.9, (n, 3)).astype(np.float32)
    comp = rng.integers(0, 4, n).astype(np.uint8)
    q = rng.normal(size=(iters, n, 4)).astype(np.float32)
    q[..., 3] = rng.uniform(0, 1, (iters, n))
    w = O.World(V, T, I, std_dev=(std,) * 4, t2=T2, dt=DT, permeability=0.4, n_cubes=n_cubes)
    return (V, T, I), w, pos, comp, q


# steps of half a cell, of some cells, and of boxes of thousands of cells
@pytest.mark.parametrize("std,n_cubes,n", [(0.02, 20, 3000), (0.08, 50, 777), (0.4, 50, 130),
                                           (0.05, 1, 65)])
def test_soup_matches_oracle(std, n_cubes, n):
    print(f"case ref soup std {std} cubes {n_cubes} spins {n}", flush=True)
    iters = 12
    (V, T, I), w, pos, comp, q = soup_case(n, iters, std, n_cubes, 7)
    grad, pc = np.array([0.02, -0.01, 0.03], np.float32), np.float32(1.5)
    st = O.State(pos, comp=comp, fiber=np.full(n, D.NO_FIBER, np.uint16))
    to = O.integrate(w, st, iters, rng=O.RNG_INJECT, inject=q, grad=grad, phase_constant=pc,
                     trace=True)
    sub = D.Substrate(V, T, I, n_cubes=n_cubes, device=n % 2 == 0)
    for trace in (True, False):  # 64 spins a wave, and fewer
        sim = D.Simulation(sub, n, dt=DT, std_dev=(std,) * 4, t2=T2, permeability=0.4,
                           mode=D.MODE_REFERENCE)
        sim.set_state(pos=pos, comp=comp)
        tg = sim.integrate_injected(grad, pc, q, trace=trace)
        if trace:
            np.testing.assert_array_equal(tg, to)
        s = sim.get_state()
        np.testing.assert_array_equal(s["pos"], st.pos)
        np.testing.assert_array_equal(s["mag"], st.mag)
        np.testing.assert_array_equal(s["phase"], st.phase)
        np.testing.assert_array_equal(s["comp"], st.comp)
        sim.close()
    assert (to[..., 2] > 0).sum() > 20
    sub.close()


def test_lists_read_through_the_triangle_index():
    # a grid without the records by list entry of the reference mode's own
    (V, T, I), _, pos, comp, q = soup_case(777, 10, 0.1, 1, 9)
    w = O.World(V, T, I, std_dev=(0.1,) * 4, t2=T2, dt=DT, permeability=0.4, **AABB)
    st = O.State(pos, comp=comp, fiber=np.full(777, D.NO_FIBER, np.uint16))
    to = O.integrate(w, st, 10, rng=O.RNG_INJECT, inject=q, trace=True)
    sub = D.Substrate(V, T, I, device=True, **AABB)
    sim = D.Simulation(sub, 777, dt=DT, std_dev=(0.1,) * 4, t2=T2, permeability=0.4,
                       mode=D.MODE_REFERENCE)
    sim.set_state(pos=pos, comp=comp)
    np.testing.assert_array_equal(
        sim.integrate_injected(np.zeros(3, np.float32), 0.0, q, trace=True), to)
    assert (to[..., 2] > 0).sum() > 20
    sim.close()
    sub.close()


def test_endless_step_among_others():
    from test_oracle_pins import _shared_diagonal_case
    env, pos, q = _shared_diagonal_case()
    n = 70
    rng = np.random.default_rng(3)
    P = rng.uniform(-0.9, 0.9, (n, 3)).astype(np.float32)
    Q = rng.normal(size=(1, n, 4)).astype(np.float32)
    Q[..., 3] = 0.5
    P[37], Q[0, 37] = pos[0], q[0, 0]
    w = O.World(env["vertices"], env["triangles"], env["tri_info"], std_dev=env["std_dev"],
                t2=env["t2"], dt=DT, permeability=0.0)
    st = O.State(P, comp=np.zeros(n, np.uint8), fiber=np.full(n, D.NO_FIBER, np.uint16))
    to = O.integrate(w, st, 1, rng=O.RNG_INJECT, inject=Q, trace=True)
    sub = D.Substrate(env["vertices"], env["triangles"], env["tri_info"])
    sim = D.Simulation(sub, n, dt=DT, std_dev=env["std_dev"], t2=env["t2"], mode=D.MODE_REFERENCE)
    sim.set_state(pos=P, comp=np.zeros(n, np.uint8), fiber=np.full(n, D.NO_FIBER, np.uint16))
    sim.integrate_injected(np.zeros(3, np.float32), 0.0, Q)
    with pytest.raises(D.DsimError) as e:
        sim.sync()
    assert e.value.code == -5
    s = sim.get_state()
    other = np.arange(n) != 37
    np.testing.assert_array_equal(s["pos"][other], st.pos[other])
    # the oracle stops after 100000 collisions, the device after 4096: both even,
    # and the loop's period is two
    assert to[0, 37, 2] == 100000
    np.testing.assert_array_equal(s["pos"][37], st.pos[37])
    sim.close()
    sub.close()
