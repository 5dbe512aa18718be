"""The physical-mode walk over triangle soups (random sizes and orientations,
long thin and degenerate triangles, coplanar pairs in either vertex order) on
every kind of grid, against the oracle on injected steps bit for bit: the
search lists' paired entries and facet bounds and the clearance shortcut may
drop no hit.  And walks of few spins, whose waves hold fewer spins each,
against the counting build, whose waves hold 64."""
import numpy as np
import pytest

import oracle as O
from dsim_amd import lib as D

pytestmark = pytest.mark.gpu

STD, T2, DT = (0.05, 0.04, 0.03, 0.05), (80.0, 70.0, 7.5, 70.0), 0.005


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if D.device_count() == 0:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")


def _soup(n, seed):
    rng = np.random.default_rng(seed)
    V, T = [], []
    for k in range(n):
        c = rng.uniform(-1.0, 1.0, 3)
        a, b = rng.normal(size=(2, 3))
        a *= np.exp(rng.uniform(np.log(0.02), np.log(2.0))) / np.linalg.norm(a)
        b *= np.exp(rng.uniform(np.log(0.02), np.log(0.5))) / np.linalg.norm(b)
        if k % 3 == 0:      # walls along z, as the prisms'
            a, b = np.array([0.0, 0.0, 2.5]), np.array([b[0], b[1], 0.0])
            c[2] = -1.25
        q = len(V)
        if k % 7 == 3:      # degenerate
            V += [c, c + a, c + 0.5 * a]
            T.append([q, q + 1, q + 2])
            continue
        V += [c, c + a, c + a + b, c + b]
        T.append([q, q + 1, q + 2])
        if k % 2 == 0:      # a coplanar pair, sharing the first vertex or not
            T.append([q, q + 2, q + 3] if k % 4 == 0 else [q + 2, q + 3, q])
    T = np.array(T, np.uint32)
    I = np.stack([np.arange(len(T)) % 50, np.zeros(len(T), int), T[:, 0]], 1).astype(np.uint32)
    return np.array(V, np.float32), T, I


GRIDS = {
    "aabb-3d": dict(grid="aabb", dims=(24, 20, 16), lo=(-1.3,) * 3, cell=(2.6 / 24, 2.6 / 20, 2.6 / 16),
                    eps=1e-5),
    "aabb-plane": dict(grid="aabb", dims=(45, 41, 1), lo=(-1.3,) * 3, cell=(2.6 / 45, 2.6 / 41, 2.6),
                       eps=1e-5),
    "aabb-one-cell": dict(grid="aabb", dims=(1, 1, 1), lo=(-1.3,) * 3, cell=(2.6,) * 3, eps=1e-5),
    "tribox-3d": dict(grid="tribox", dims=(24, 20, 16), lo=(-1.3,) * 3,
                      cell=(2.6 / 24, 2.6 / 20, 2.6 / 16), eps=1e-5),
    "reference": dict(grid="reference", n_cubes=20),
}


@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("grid", sorted(GRIDS))
def test_soup_matches_oracle(grid, boundary):
    print(f"case soup {grid} boundary {boundary}", flush=True)
    V, T, I = _soup(240, 3)
    g = GRIDS[grid]
    og = dict(GRIDS["aabb-3d" if g["grid"] == "tribox" else grid])
    if og["grid"] == "reference":
        og = dict(grid="reference", n_cubes=20)
    n, iters = 2000, 60
    w = O.World(V, T, I, std_dev=STD, t2=T2, dt=DT, permeability=0.3, test=1, traversal=1,
                transitions=1, boundary=boundary, **og)
    sub = D.Substrate(V, T, I, device=grid != "aabb-plane", **g)  # one of them built on the host
    sim = D.Simulation(sub, n, dt=DT, std_dev=STD, t2=T2, permeability=0.3, mode=D.MODE_PHYSICAL,
                       boundary=boundary, seed=5)
    rng = np.random.default_rng(11)
    pos = rng.uniform(-0.95, 0.95, (n, 3)).astype(np.float32)
    comp = rng.integers(0, 3, n).astype(np.uint8)
    q = rng.normal(size=(iters, n, 4)).astype(np.float32)
    q[..., 3] = rng.uniform(0, 1, (iters, n))
    st = O.State(pos, comp=comp, fiber=np.full(n, D.NO_FIBER, np.uint16), moment=True)
    to = O.integrate(w, st, iters, rng=O.RNG_INJECT, inject=q, weight=1.0, trace=True)
    sim.set_state(pos=pos, comp=comp)
    sim.moment_reset()
    tg = sim.integrate_moment_injected(1.0, q, trace=True)
    cols = [0, 1, 2, 4] if g["grid"] == "tribox" else [0, 1, 2, 3, 4]  # 3: the oracle's cell
    np.testing.assert_array_equal(tg[..., cols], to[..., cols])
    s = sim.get_state()
    np.testing.assert_array_equal(s["pos"], st.pos)
    np.testing.assert_array_equal(s["mag"], st.mag)
    assert (to[..., 2] > 0).sum() > 5000
    sim.close()
    sub.close()


@pytest.mark.parametrize("n", [1, 5, 63, 64, 65, 1000, 16384, 16385, 70001])
def test_few_spins_walk_as_in_full_waves(n):
    print(f"case few spins {n}", flush=True)
    V, T, I = _soup(240, 4)
    sub = D.Substrate(V, T, I, device=True, **GRIDS["aabb-plane"])
    out = []
    for counting in (False, True):
        sim = D.Simulation(sub, n, dt=DT, std_dev=STD, t2=T2, permeability=0.3,
                           mode=D.MODE_PHYSICAL, boundary=D.BOUNDARY_PERIODIC, seed=n)
        sim.init_uniform(1.0)
        sim.moment_reset()
        if counting:
            sim.walk_stats(True)
        sim.integrate_moment(1.0, 50)
        out.append((sim.get_state(), sim.get_moment()[0]))
        sim.close()
    sub.close()
    for k in ("pos", "mag", "comp", "fiber"):
        np.testing.assert_array_equal(out[0][0][k], out[1][0][k])
    np.testing.assert_array_equal(out[0][1], out[1][1])
