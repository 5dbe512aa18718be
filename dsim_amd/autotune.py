"""Launch-shape autotuner for the step kernel.

The grid cell edge sets how many candidate triangles a step tests (small
cells: few candidates but more cells per step; large cells: long lists), and
the spatial-sort interval sets how coherent a wavefront's cells stay.  Both
depend on the substrate, so they are chosen by timing short runs of the real
workload on the device: every candidate builds its grid, walks all spins for
a few hundred steps, and the fastest (steps per second from HIP events on the
step kernels) wins.
"""
from __future__ import annotations

import time

import numpy as np

from . import lib as D
from . import substrate as S


def launch_steps(sort_interval):
    """Steps per step-kernel launch for a reorder interval: one launch per
    interval (at least 256 steps), 1024 without reordering.  A launch ends when
    its slowest lane finishes, so longer launches leave lanes idle less often."""
    if sort_interval == 0:
        return 1024
    return max(256, sort_interval)


def make_sim(env, n, *, sort_interval, steps_per_launch=0, seed=None, device_build=True):
    g = env["grid"]
    cfg = env["cfg"]
    sub = D.Substrate(env["vertices"], env["triangles"], env["tri_info"], grid="aabb",
                      dims=g["dims"], lo=g["lo"], cell=g["cell"], eps=g["eps"],
                      device=device_build)
    sim = D.Simulation(sub, n, dt=cfg.dt, std_dev=env["std_dev"], t2=env["t2"],
                       permeability=env["permeability"], mode=D.MODE_PHYSICAL,
                       boundary=D.BOUNDARY_PERIODIC, rng=D.RNG_PHILOX,
                       seed=cfg.seed if seed is None else seed, sort_interval=sort_interval,
                       steps_per_launch=steps_per_launch)
    return sub, sim


def time_steps(sim, steps, warm=64):
    sim.moment_reset()
    sim.integrate_moment(1.0, warm)
    sim.sync()
    sim.step_timing_reset()
    sim.integrate_moment(1.0, steps)
    sim.sync()
    ms, _ = sim.step_timing()
    return ms / 1e3


# Reorder intervals tried.  4096 steps was measured no faster than 2048 on the
# 1e6-spin, 2000-axon substrate (47.8 against 47.0 ms of step kernel per 1000
# steps), but within the tie tolerance it would be picked as the longer one.
SORTS = (0, 256, 512, 1024, 2048)


def tune(cfg, axons, n, *, cells_um=(0.15, 0.2, 0.25), sorts=SORTS,
         steps=1024, warm=320, tie_tol=0.01, log=None):
    """Returns (best dict, all results).  Each result: cell_um, sort_interval,
    spin-steps/s, grid dims.  Among the candidates within tie_tol of the
    fastest (run-to-run timing noise), the one with the longest reorder
    interval, then the largest cell (fewer reorders, smaller grid) is chosen,
    so that repeated runs settle on the same configuration.  Each candidate
    launches launch_steps(sort) steps at a time, its warm-up runs past the
    first reorder keyed by measured search rates, and it is timed over at least
    `steps` and two of its reorder intervals (whole launches and their
    reorders)."""
    results = []
    for h in cells_um:
        env = S.build(cfg, cell_um=h, axons=axons)
        for srt in sorts:
            t0 = time.perf_counter()
            sub, sim = make_sim(env, n, sort_interval=srt, steps_per_launch=launch_steps(srt))
            sim.init_uniform(1.0)
            sim.label(env["xmax"], env["xmax"], env["xmax"])
            # warm up past the first reorder keyed by measured search rates
            timed = max(steps, 2 * srt)
            sec = time_steps(sim, timed, warm=max(warm, srt + 64))
            rate = n * timed / sec
            r = dict(cell_um=h, sort_interval=srt, rate=rate, grid=list(env["grid"]["dims"]),
                     setup_s=time.perf_counter() - t0 - sec)
            results.append(r)
            if log:
                log(f"autotune cell {h:.3f} um sort {srt}: {rate:.3e} spin-steps/s "
                    f"(grid {r['grid']})")
            sim.close()
            sub.close()
    return pick(results, tie_tol), results


def pick(results, tie_tol=0.01):
    """The candidate to use: among those within tie_tol of the fastest rate,
    the longest reorder interval, then the largest cell."""
    top = max(r["rate"] for r in results)
    near = [r for r in results if r["rate"] >= (1.0 - tie_tol) * top]
    return max(near, key=lambda r: (r["sort_interval"], r["cell_um"]))
