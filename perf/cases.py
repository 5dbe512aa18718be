"""Timed cases of the simulate path through its public entry points.

A case is a dict of plain values.  `listed()` names twelve; `draw()` gives
more of the same ranges; `prepare()` makes what a program holds before the
call (substrate, simulation handle, gradients), `run()` is one pass, `work()`
what a pass cannot do without, `exact()` the outputs in 64 bits where they
have a closed form.

The kinds of work:

  acquisition  one shared-gradient acquisition: every spin walks the PGSE
               sequence once (moment reset, four lobes), then one signal per
               gradient line; the benchmark's own step
  line         one gradient line the way the reference's sequencer plays it:
               spins drawn and labelled, four lobes of the per-step phase path,
               the signal, the final state read back
  updates      the drop-in path (reference semantics, 50^3 grid, MWC draws) in
               update() calls of a few steps, signal and state read back
  label        a fresh set of spins drawn, labelled and read back
  waveforms    phases of arbitrary gradient waveforms over one walk, the
               waveforms handed over for this acquisition
  served       a queue of requests on resident substrates through the server
  readout      signals from moments the caller holds on the device

Meshes: "small" is the 16-axon packing with caps; "tile<k>" repeats a
125-axon periodic packing of the at-scale statistics k times along x and y
(tile4: 2000 axons, about 280,000 triangles); "bundles<n>" is two crossing
bundles of n axons over an exact-membership grid; "water" has no triangles.
"""
import ctypes
import dataclasses
import functools
import math

import numpy as np
import torch

from dsim_amd import batched as B
from dsim_amd import crossing as X
from dsim_amd import lib as D
from dsim_amd import phase as PH
from dsim_amd import serve as SV
from dsim_amd import substrate as S

GAMMA = 42576.0
DT = 0.005
PC = np.float32(2 * np.pi * GAMMA * DT)


def listed():
    return [
        # the headline workload: 1e6 spins, 2000 permeable axons, PGSE 10/40/60
        # ms (12,000 steps), 64 directions and b = 0, spins reordered
        {"name": "acquisition-1m", "kind": "acquisition", "mesh": "tile4", "spins": 1_000_000,
         "steps": 12000, "lines": 65, "sort": 2048},
        # the small configuration as it stands: 1e4 spins, 16 axons, 7 lines
        {"name": "acquisition-10k", "kind": "acquisition", "mesh": "small", "spins": 10_000,
         "steps": 12000, "lines": 7, "sort": 0},
        # crossing bundles: a 3-D grid with indirect records, a ragged spin
        # count that does not fill the device
        {"name": "acquisition-bundles", "kind": "acquisition", "mesh": "bundles200",
         "spins": 50_001, "steps": 2400, "lines": 33, "sort": 0},
        # one line of the reference's sequence (every line draws and labels its
        # spins anew), phase path in a periodic voxel, spins reordered
        {"name": "line-100k", "kind": "line", "mesh": "tile2", "spins": 100_003, "steps": 2000,
         "sort": 512},
        # drop-in update() of ten steps on a thousand spins: launch latency
        {"name": "update-1k", "kind": "updates", "mesh": "small", "spins": 1000, "updates": 1,
         "iters": 10},
        # the command line's size: 20,000 spins, ten steps an update
        {"name": "updates-20k", "kind": "updates", "mesh": "small", "spins": 20_000,
         "updates": 20, "iters": 10},
        # the reference semantics at a million spins
        {"name": "updates-1m", "kind": "updates", "mesh": "small", "spins": 1_000_000,
         "updates": 5, "iters": 100},
        # labelling a million spins on the at-scale substrate
        {"name": "label-1m", "kind": "label", "mesh": "tile4", "spins": 1_000_000},
        # many waveforms over many spins: the matrix-core path
        {"name": "waveforms-500k", "kind": "waveforms", "mesh": "small", "spins": 500_000,
         "waveforms": 1024, "steps": 2048, "chunk": 64, "buffer": 1024},
        # a calibration run in open water, sizes that fill no tile
        {"name": "waveforms-water", "kind": "waveforms", "mesh": "water", "spins": 4099,
         "waveforms": 200, "steps": 320, "chunk": 64, "buffer": 320},
        # a queue of mixed requests on resident crossing substrates
        {"name": "served-24", "kind": "served", "substrates": 4, "requests": 24, "spins": 60_000,
         "steps": 1500},
        # the allocation-free readout of a million spins at the headline's lines
        {"name": "readout-1m", "kind": "readout", "spins": 1_000_000, "lines": 65,
         "balanced": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["acquisition", "acquisition", "line", "updates", "label", "waveforms",
                       "served", "readout"])
    mesh = rng.choice(["small", "tile1", "tile2", "tile3", "tile4"])
    if kind in ("acquisition", "line"):
        if rng.random() < 0.3:
            mesh = "bundles%d" % rng.choice([50, 100, 200, 400])
        n = _log_int(rng, 1000, 1_000_000)
        steps = _log_int(rng, 300, min(12000, max(400, 1.5e9 / n)))
        sort = rng.choice([0, 256, 512, 2048])
        c = {"kind": kind, "mesh": mesh, "spins": n, "steps": steps, "sort": sort}
        return dict(c, lines=rng.randint(7, 65)) if kind == "acquisition" else c
    if kind == "updates":
        n = _log_int(rng, 1000, 1_000_000)
        return {"kind": kind, "mesh": "small", "spins": n, "updates": rng.randint(1, 20),
                "iters": rng.choice([5, 10, 10, 20, 25])}
    if kind == "label":
        return {"kind": kind, "mesh": rng.choice([mesh, "bundles100", "bundles400"]),
                "spins": _log_int(rng, 1000, 1_000_000)}
    if kind == "waveforms":
        chunk = 32 * rng.choice([1, 2, 2, 4])
        buffer = chunk * rng.randint(1, max(1, 1024 // chunk))
        return {"kind": kind, "mesh": rng.choice(["small", "small", "water", "tile1"]),
                "spins": _log_int(rng, 1000, 500_000), "waveforms": _log_int(rng, 20, 1024),
                "steps": 32 * rng.randint(3, 40), "chunk": chunk, "buffer": buffer}
    if kind == "served":
        return {"kind": kind, "substrates": rng.randint(1, 4), "requests": rng.randint(4, 24),
                "spins": _log_int(rng, 15_000, 100_000), "steps": rng.randint(600, 1500)}
    return {"kind": "readout", "spins": _log_int(rng, 1000, 1_000_000),
            "lines": rng.randint(1, 128), "balanced": rng.random() < 0.7}


# ---- substrates ------------------------------------------------------------ #

@functools.lru_cache(maxsize=None)
def _mesh(name):
    """Host mesh, grid and physics of a named substrate (what a program reads
    from its files once)."""
    if name == "small":
        e = S.build(S.SMALL, cell_um=0.2, axons=S.pack(S.SMALL))
    elif name.startswith("tile"):
        k = int(name[4:])
        cfg = dataclasses.replace(S.SCALE, name=name, n_axons=125)
        a = S.pack(cfg)
        at = [a.centers + a.voxel * np.array([i, j]) for i in range(k) for j in range(k)]
        e = S.build(cfg, cell_um=0.2, axons=S.Axons(np.concatenate(at), np.tile(a.radii, k * k),
                                                    a.voxel * k, a.intra_fraction))
    elif name == "water":
        sd = np.float32(math.sqrt(2 * 2.0 * DT) / 10.0)  # a 20 um voxel, 2 um^2/ms
        return dict(V=np.zeros((0, 3), np.float32), T=np.zeros((0, 3), np.uint32),
                    I=np.zeros((0, 3), np.uint32), scale=10.0, extent=(1.0,) * 3,
                    grid=dict(grid="aabb", dims=(10, 10, 10), lo=(-1.0,) * 3, cell=(0.2,) * 3),
                    box=((-1.0,) * 3, (1.0,) * 3), std_dev=(sd,) * 4, t2=(np.inf,) * 4,
                    permeability=0.0)
    else:
        n = int(name[7:])
        cs = B.CrossingSet()
        cx = X.make_crossing(n, 1.0, 45.0, np.random.default_rng(n), ngon=cs.ngon)
        V, T, I, s = X.crossing_mesh(cx, cs.halo_um)
        g, _ = B.grid_for(cs, cx, 0.3 * float(np.mean(np.concatenate([cx.a_r, cx.b_r]))))
        lo, hi = X.voxel_bounds(cx)
        return dict(V=V, T=T, I=I, scale=s, extent=tuple(float(v) for v in np.abs(V).max(0)),
                    grid=dict(grid="tribox", **g), box=(tuple(lo), tuple(hi)), **B.physics(cs, s))
    g = e["grid"]
    return dict(V=e["vertices"], T=e["triangles"], I=e["tri_info"], scale=e["space_scale"],
                extent=(e["xmax"],) * 3, box=((-1.0,) * 3, (1.0,) * 3), std_dev=e["std_dev"],
                t2=e["t2"], permeability=e["permeability"],
                grid=dict(grid="aabb", dims=g["dims"], lo=g["lo"], cell=g["cell"], eps=g["eps"]))


def _physical(mesh, n, seed, sort=0):
    m = _mesh(mesh)
    sub = D.Substrate(m["V"], m["T"], m["I"], device=True, **m["grid"])
    sim = D.Simulation(sub, n, dt=DT, std_dev=m["std_dev"], t2=m["t2"],
                       permeability=m["permeability"], mode=D.MODE_PHYSICAL,
                       boundary=D.BOUNDARY_PERIODIC, rng=D.RNG_PHILOX, seed=seed,
                       sort_interval=sort, steps_per_launch=max(256, sort) if sort else 0,
                       voxel=m["box"])
    return m, sub, sim


def _draw_spins(m, sim):
    sim.init_box(*m["box"])
    return sim.label(*m["extent"])


def _lobes(steps):
    """PGSE lobes in the proportions of delta/Delta/TE = 10/40/60 ms."""
    L, R = steps // 6, steps // 6
    B_ = steps - L - R
    return [(1.0, L), (0.0, B_ - L), (-1.0, L), (0.0, R)]


def _lines(steps, lines, scale, b=1.0):
    """b = 0 and lines - 1 directions on three shells, gradScaled units."""
    L, B_ = steps // 6 * DT, (steps - 2 * (steps // 6)) * DT
    g = [np.zeros(3)]
    for k, d in enumerate(S.fibonacci_directions(max(1, lines - 1))):
        g.append(d * S.gradient_amplitude(b * (1 + k % 3), L, B_))
    return (np.array(g[:lines]) * 1e-9 * scale).astype(np.float32)


def _state(sim):
    s = sim.get_state()
    return {"pos": s["pos"], "mag": s["mag"], "phase": s["phase"],
            "comp": s["comp"].astype(np.int32), "fiber": s["fiber"].astype(np.int32)}


# ---- cases ------------------------------------------------------------------ #

def prepare(case, seed):
    kind = case["kind"]
    if kind == "acquisition":
        m, sub, sim = _physical(case["mesh"], case["spins"], seed, case["sort"])
        _draw_spins(m, sim)
        return dict(case, sub=sub, sim=sim, lobes=_lobes(case["steps"]),
                    grads=_lines(case["steps"], case["lines"], m["scale"]))
    if kind == "line":
        m, sub, sim = _physical(case["mesh"], case["spins"], seed, case["sort"])
        return dict(case, m=m, sub=sub, sim=sim, lobes=_lobes(case["steps"]),
                    grad=_lines(case["steps"], 2, m["scale"])[1])
    if kind == "updates":
        m = _mesh(case["mesh"])
        sub = D.Substrate(m["V"], m["T"], m["I"], device=True)  # the reference's 50^3 grid
        sim = D.Simulation(sub, case["spins"], dt=DT, std_dev=m["std_dev"], t2=m["t2"],
                           permeability=m["permeability"], mode=D.MODE_REFERENCE,
                           boundary=D.BOUNDARY_CLAMP, rng=D.RNG_MWC, seed=seed)
        sim.init_uniform(1.0)
        sim.label(*m["extent"])
        grad = np.array([0.0, 61.7e-9 * m["scale"], 0.0], np.float32)
        return dict(case, sub=sub, sim=sim, grad=grad)
    if kind == "label":
        m, sub, sim = _physical(case["mesh"], case["spins"], seed)
        return dict(case, m=m, sub=sub, sim=sim)
    if kind == "waveforms":
        m, sub, sim = _physical(case["mesh"], case["spins"], seed)
        _draw_spins(m, sim)
        return dict(case, sub=sub, sim=sim, grads=_waveforms(case, seed, m["scale"]))
    if kind == "served":
        return _prepare_served(case, seed)
    return _prepare_readout(case, seed)


def _waveforms(case, seed, scale):
    return PH.random_waveforms(case["waveforms"], case["steps"], seed) * np.float32(1e-9 * scale)


def _prepare_served(case, seed):
    rng = np.random.default_rng(seed)
    srv = SV.Server(100 << 30)
    subs = []
    for n in (50, 100, 200, 400)[:case["substrates"]]:
        m = _mesh("bundles%d" % n)
        sub = D.Substrate(m["V"], m["T"], m["I"], device=True, **m["grid"])
        subs.append((m, sub, srv.add_substrate(sub)))
    reqs = []
    for k in range(case["requests"]):
        m, _, i = subs[int(rng.integers(len(subs)))]
        n = int(round(math.exp(rng.uniform(math.log(1e4), math.log(case["spins"])))))
        steps = case["steps"]
        lobes = _lobes(steps)
        reqs.append(dict(substrate=i, n_spins=n, seed=seed * 1000 + k, dt=DT,
                         std_dev=m["std_dev"], t2=m["t2"], permeability=m["permeability"],
                         lobes=lobes, grads=_lines(steps, 7 + 8 * (k % 8), m["scale"]),
                         phase_constant=PC, label_extent=m["extent"], voxel=m["box"]))
    return dict(case, srv=srv, subs=subs, reqs=reqs)


def _prepare_readout(case, seed):
    n, k = case["spins"], case["lines"]
    g = torch.Generator(device="cuda").manual_seed(seed)

    def uniform(*shape):
        return torch.rand(*shape, generator=g, device="cuda")

    # end of an acquisition: decayed magnitudes, a third of the spins outside
    # the axons, moments of free and hindered walks of 12,000 steps
    u = uniform(n)
    comp = torch.where(u < 0.3, 0, torch.where(u < 0.95, 1, 2)).to(torch.int32)
    mag = 0.4 + 0.1 * uniform(n)
    mom = torch.randn(3, n, generator=g, device="cuda") * 1500.0
    x0 = 2.0 * uniform(3, n) - 1.0
    grads = _lines(12000, k, 53.95)
    return dict(case, mag=mag, mom=mom, x0=x0, label=comp | (65535 << 8),
                grads=torch.from_numpy(grads).cuda(), wsum=0.0 if case["balanced"] else 250.0,
                out=torch.zeros(k, 5, dtype=torch.float64, device="cuda"))


def _read(f, *args):
    """A readout.  A step whose collision loop does not end (a segment on the
    diagonal of two coplanar triangles in the reference semantics, about one
    in 1e9) is stopped and reported once by the next call that waits; the
    state stays valid and the program reads again."""
    try:
        return f(*args)
    except D.DsimError as e:
        if e.code != -5:
            raise
        return f(*args)


def run(state):
    kind = state["kind"]
    if kind == "acquisition":
        sim = state["sim"]
        sim.moment_reset()
        for w, k in state["lobes"]:
            sim.integrate_moment(w, k)
        return {"signals": _read(sim.signal_moment, state["grads"], PC)}
    if kind == "line":
        sim = state["sim"]
        ambiguous = _draw_spins(state["m"], sim)
        for w, k in state["lobes"]:
            sim.integrate(np.float32(w) * state["grad"], PC, k)
        return {"ambiguous": ambiguous, "signal": _read(sim.signal), "state": _state(sim)}
    if kind == "updates":
        sim = state["sim"]
        for _ in range(state["updates"]):
            sim.integrate(state["grad"], PC, state["iters"])
        return {"signal": _read(sim.signal), "state": _state(sim)}
    if kind == "label":
        sim = state["sim"]
        return {"ambiguous": _draw_spins(state["m"], sim), "state": _state(sim)}
    if kind == "waveforms":
        sim = state["sim"]
        sim.moment_reset()
        wf = PH.Waveforms(sim, state["grads"], PC, chunk_steps=state["chunk"],
                          buffer_steps=state["buffer"])
        # the handle's arrays are cleared on the default stream, its walk runs
        # on its own: threadSync in between
        D.check(D.lib().dsim_thread_sync())
        wf.run(state["steps"])
        out = {"signal": wf.signal()}
        if state["spins"] * state["waveforms"] <= 4_000_000:
            out["phase"] = wf.phase()[0]
        wf.close()
        return out
    if kind == "served":
        srv = state["srv"]
        tickets = [srv.submit(**q) for q in state["reqs"]]
        srv.run_until_idle()
        return [srv.result(t)[0] for t in tickets]
    f = _nalloc()
    rc = f(state["spins"], state["mag"].data_ptr(), state["mom"].data_ptr(),
           state["x0"].data_ptr(), state["wsum"], state["label"].data_ptr(), state["lines"],
           state["grads"].data_ptr(), float(PC), state["out"].data_ptr(), None)
    D.check(rc)
    return state["out"]


@functools.lru_cache(maxsize=None)
def _nalloc():
    f = D.lib().dsim_signal_moment_nalloc
    p = ctypes.c_void_p
    f.argtypes = [ctypes.c_uint32, p, p, p, ctypes.c_float, p, ctypes.c_uint32, p,
                  ctypes.c_float, p, p]
    f.restype = ctypes.c_int
    return f


def work(case):
    """Walks: the benchmark's work model (50 + 7 a moment channel + 45 a
    triangle whose box meets the step's + 21 a hit: 104 operations a spin-step
    at the at-scale densities) and the spins' state once in and once out.
    Waveforms: three bf16 products a multiply-add.  Readout and signals: about
    40 operations of a 64-bit sine and cosine a spin and line."""
    n = case.get("spins", 0)
    kind = case["kind"]
    state = 2 * 68 * n  # position, magnitude, label, displacement, moments, x0
    if kind == "acquisition":
        return {"bytes": state + 20 * n, "flops": 104.0 * n * case["steps"] + 40.0 * n * case["lines"]}
    if kind == "line":
        return {"bytes": 2 * 28 * n, "flops": 104.0 * n * case["steps"]}
    if kind == "updates":
        return {"bytes": 2 * 32 * n, "flops": 104.0 * n * case["updates"] * case["iters"]}
    if kind == "label":
        return {"bytes": 24 * n + 12 * len(_mesh(case["mesh"])["V"]), "flops": 104.0 * n}
    if kind == "waveforms":
        k = 3 * case["steps"]
        return {"bytes": 4.0 * case["waveforms"] * k + state + 8.0 * case["waveforms"],
                "flops": 6.0 * n * case["waveforms"] * k + 104.0 * n * case["steps"]}
    if kind == "served":
        mean = (n - 1e4) / math.log(n / 1e4)
        total = case["requests"] * mean
        return {"bytes": 2 * 68 * total, "flops": 104.0 * total * case["steps"]}
    return {"bytes": 32.0 * n + 52.0 * case["lines"], "flops": 40.0 * n * case["lines"]}


# ---- 64-bit values ---------------------------------------------------------- #

def _philox(c, k0, k1):
    """Philox4x32-10 over arrays of counter words."""
    c = [np.asarray(x, np.uint64) for x in c]
    low = np.uint64(0xFFFFFFFF)
    for r in range(10):
        a, b = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        ka, kb = (k0 + r * 0x9E3779B9) & 0xFFFFFFFF, (k1 + r * 0xBB67AE85) & 0xFFFFFFFF
        c = [(b >> np.uint64(32)) ^ c[1] ^ np.uint64(ka), b & low,
             (a >> np.uint64(32)) ^ c[3] ^ np.uint64(kb), a & low]
    return c


def _unit(w):
    return ((w >> np.uint64(9)).astype(np.float64) + 0.5) * 2.0 ** -23


def _magnitudes(re, im, comp):
    """|sum| / count over all spins and per compartment, [line, 5]."""
    out = np.zeros((re.shape[1], 5))
    for c in range(-1, 4):
        sel = slice(None) if c < 0 else comp == c
        count = len(comp) if c < 0 else int(sel.sum())
        if count:
            out[:, c + 1] = np.hypot(re[sel].sum(0), im[sel].sum(0)) / count
    return out


def exact(case, seed):
    """The readout of given moments, and the phases of free walkers.  A walk
    among membranes has no 64-bit value of its own: a spin whose last bit
    differs meets another wall soon after."""
    if case["kind"] == "readout":
        s = _prepare_readout(case, seed)
        mag, mom, x0 = (s[k].double().cpu().numpy() for k in ("mag", "mom", "x0"))
        comp = (s["label"].cpu().numpy() & 0xFF)
        g = s["grads"].double().cpu().numpy()
        out = np.zeros((case["lines"], 5))
        for j in range(case["lines"]):
            ph = float(PC) * (g[j] @ (mom + s["wsum"] * x0))
            out[j] = _magnitudes((mag * np.cos(ph))[:, None], (mag * np.sin(ph))[:, None], comp)[0]
        return out
    if case["kind"] == "waveforms" and case["mesh"] == "water":
        n, steps, W = case["spins"], case["steps"], case["waveforms"]
        if n * W * steps > 4e9 or n * steps > 2e7:
            return None
        m = _mesh("water")
        i = np.arange(n)
        x0 = np.stack([2.0 * (_unit(w) - 0.5) for w in _philox([i, 0 * i, 0 * i, 0 * i + 2],
                                                               seed & 0xFFFFFFFF, seed >> 32)[:3]])
        t = np.arange(steps)[:, None] + 0 * i
        u = [_unit(w) for w in _philox([i + 0 * t, t, 0 * t, 0 * t], seed & 0xFFFFFFFF, seed >> 32)]
        r1, r2 = np.sqrt(-2 * np.log(u[0])), np.sqrt(-2 * np.log(u[2]))
        d = np.stack([r1 * np.cos(2 * np.pi * u[1]), r1 * np.sin(2 * np.pi * u[1]),
                      r2 * np.cos(2 * np.pi * u[3])], 1) * float(m["std_dev"][0])
        walk = np.cumsum(d, 0)                                       # [steps, 3, n]
        g = _waveforms(case, seed, m["scale"]).astype(np.float64) * float(PC)  # [steps, W, 3]
        ph = np.ascontiguousarray(walk.transpose(2, 0, 1)).reshape(n, -1) @ \
            np.ascontiguousarray(g.transpose(0, 2, 1)).reshape(-1, W)
        total = ph + x0.T @ g.sum(0).T
        out = {"signal": _magnitudes(np.cos(total), np.sin(total), np.zeros(n, int))}
        if n * W <= 4_000_000:
            out["phase"] = ph
        return out
    return None
