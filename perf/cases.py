"""The work that users of this package have it do, as cases that can be timed.

Three kinds, each through the public entry points of koral_zig_amd:

  run     a PUFFY run advanced by some CFL steps (Sim.step, Sim.step_many, a
          captured batch replayed, or the single passes of a step driven by
          the caller), after which the caller takes the state out: what a
          driver does between two outputs.  The run keeps going from pass to
          pass.
  batch   independent implicit radiation-gas solves from host arrays
          (ImplicitBatch.solve and .get; the inputs are loaded beforehand).
  device  the same solve over the caller's own device arrays
          (kz_implicit_solve_noalloc), as serving loops call it.

Sizes are the run server's five grids, the 384x360 torus, 3D wedges, the
independent-cell batch, and odd sizes between.  All of it is FP64.

`exact` has no values: the outputs are FP64 already, and the same quantities
from plain array code would be a second implementation of the whole solver.
"""
import ctypes
import functools
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

PACKAGE = Path(__file__).resolve().parent.parent / "koral-zig_amd"
if "koral_zig_amd" not in sys.modules:
    _spec = importlib.util.spec_from_file_location("koral_zig_amd", PACKAGE / "__init__.py",
                                                   submodule_search_locations=[str(PACKAGE)])
    _module = importlib.util.module_from_spec(_spec)
    sys.modules["koral_zig_amd"] = _module
    _spec.loader.exec_module(_module)
from koral_zig_amd import abi_types as T  # noqa: E402
from koral_zig_amd import hip, host, workloads  # noqa: E402


def _run(name, nx, ny, steps, nz=1, spin=0.0, drive="many", physics="default"):
    return {"name": name, "kind": "run", "nx": nx, "ny": ny, "nz": nz, "spin": spin, "steps": steps, "drive": drive,
            "physics": physics}


def listed():
    return [
        # the smallest run, each step taken and looked at by itself (a debugger, a coupled code)
        _run("step_64x64", 64, 64, 1, drive="step"),
        # one resident run of a server: batches of ten steps replayed from a graph
        _run("replay_128x96", 128, 96, 10, spin=0.5, drive="replay"),
        # a driver in another language that calls the passes of a step itself; odd extents
        _run("passes_211x173", 211, 173, 4, drive="passes"),
        # the reference's runtime options: ZAMO-frame floor, synchrotron bridge, both reduced orders
        _run("options_192x192", 192, 192, 20, spin=0.9, physics="options"),
        # a middle-sized run of a spinning hole
        _run("run_256x256", 256, 256, 40, spin=0.9375),
        # the headline torus between two outputs
        _run("torus_384x360", 384, 360, 100),
        # the same torus as production runs it: radiative viscosity and the mimic dynamo
        _run("production_384x360", 384, 360, 50, physics="production"),
        # a small 3D wedge (a test run before the large one)
        _run("wedge_48x48x16", 48, 48, 20, nz=16, spin=0.9375),
        # a 3D wedge large enough for the persistent implicit launches
        _run("wedge_128x128x32", 128, 128, 40, nz=32, spin=0.9375),
        # a small odd batch of independent solves: latency
        {"name": "batch_4099", "kind": "batch", "cells": 4099},
        # a survey of solver states
        {"name": "batch_524288", "kind": "batch", "cells": 1 << 19},
        # a serving loop with its states already on the device
        {"name": "device_20000", "kind": "device", "cells": 20000},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choices(("2d", "3d", "batch", "device"), (6, 2, 2, 2))[0]
    if what == "batch":
        return {"kind": "batch", "cells": _log_uniform(rng, 1000, 400000)}
    if what == "device":
        return {"kind": "device", "cells": _log_uniform(rng, 200, 32768)}
    spin = round(rng.uniform(0.0, 0.95), 3)
    drive = rng.choices(("many", "step", "replay", "passes"), (5, 1, 2, 1))[0]
    steps = {"many": rng.randint(5, 60), "step": rng.randint(1, 4), "replay": rng.randint(5, 20),
             "passes": rng.randint(1, 6)}[drive]
    if what == "3d":
        return {"kind": "run", "nx": rng.randint(32, 96), "ny": rng.randint(32, 96), "nz": rng.randint(8, 24),
                "spin": spin, "steps": min(steps, 20), "drive": drive, "physics": rng.choice(("default", "options"))}
    return {"kind": "run", "nx": _log_uniform(rng, 48, 360), "ny": _log_uniform(rng, 48, 340), "nz": 1, "spin": spin,
            "steps": steps, "drive": drive, "physics": rng.choice(("default", "default", "production", "options"))}


def _grid(case):
    return T.grid_puffy(case["nx"], case["ny"], case["nz"], rmin=T.rmin_for_spin(case["spin"]))


@functools.lru_cache(maxsize=2)
def _torus(nx, ny, nz, spin):
    """Metric tables and the unperturbed torus of a grid: a program that
    starts several runs on one grid computes them once."""
    grid = T.grid_puffy(nx, ny, nz, rmin=T.rmin_for_spin(spin))
    tables = host.metric_tables(grid, dict(host.MP_PUFFY, a=spin))
    return tables, host.puffy_prepinit(grid, tables, T.physics_puffy(bh_spin=spin))


@functools.lru_cache(maxsize=1)
def _bl_tables(nx, ny, nz, spin):
    grid = T.grid_puffy(nx, ny, nz, rmin=T.rmin_for_spin(spin))
    return host.bl_tables(grid, dict(host.MP_PUFFY, a=spin))


def _physics(case, grid):
    production = case["physics"] == "production"
    ph = T.physics_puffy(radviscosity=production, dynamo=production, bh_spin=case["spin"])
    if case["physics"] == "options":
        ph.floors.b2rhofloorframe = 1
        ph.opac.synchrotron_bridge = 1
        ph.reduceorderatbh = 1
        ph.reduce_order_ix_max = host.reduce_order_ix_max(grid, dict(host.MP_PUFFY, a=case["spin"]))
        ph.reduceorderafterfixup = 1
    return ph


def _prepare_run(case, seed):
    grid = _grid(case)
    ph = _physics(case, grid)
    tables, p0 = _torus(case["nx"], case["ny"], case["nz"], case["spin"])
    sim = hip.Sim(grid, ph, tables)
    if case["physics"] == "production":
        sim.set_bl_tables(_bl_tables(case["nx"], case["ny"], case["nz"], case["spin"]))
    host.init_puffy(sim, grid, tables, ph, seed=seed, rho_u_only=case["nz"] > 1, p0=p0)
    # past the startup steps, whose timestep is a guess
    sim.step_many(3)
    sim.sync()
    if case["drive"] == "replay":
        sim.capture_steps(case["steps"])
    return {"kind": "run", "sim": sim, "steps": case["steps"], "drive": case["drive"],
            "dt": 0.1 * sim.counters()["dt"]}


def prepare(case, seed):
    if case["kind"] == "run":
        return _prepare_run(case, seed)
    n = case["cells"]
    ph = T.physics_puffy()
    pp, geom, dt = workloads.implicit_batch_inputs(
        n, seed, ph, lambda p, g: hip.radstate(p, g, ph.gam, ph.opac, 0)[:, 9])
    if case["kind"] == "batch":
        batch = hip.ImplicitBatch(n, ph)
        batch.set(pp, geom, dt)
        return {"kind": "batch", "batch": batch}
    f64 = dict(dtype=torch.float64, device="cuda")
    return {"kind": "device", "n": n, "physics": ph,
            "pp_in": torch.from_numpy(np.ascontiguousarray(pp)).cuda(),
            "geom": torch.from_numpy(np.ascontiguousarray(geom)).cuda(),
            "dt": torch.from_numpy(np.ascontiguousarray(dt)).cuda(),
            "uu": torch.empty((n, T.NV), **f64), "pp": torch.empty((n, T.NV), **f64),
            "result": torch.empty((n, T.IMPLICIT_RESULT_DTYPE.itemsize // 4), dtype=torch.int32, device="cuda"),
            "counts": torch.empty(3, dtype=torch.int64, device="cuda")}


def _passes(sim, dt):
    """One operator-split step by the single passes, in the order of a step."""
    sim.op_implicit(dt)
    sim.calc_u2p()
    sim.do_correct()
    sim.set_bc()
    sim.op_explicit(dt)
    sim.do_correct()
    sim.set_bc()


def run(state):
    if state["kind"] == "run":
        sim = state["sim"]
        if state["drive"] == "step":
            for _ in range(state["steps"]):
                sim.step()
        elif state["drive"] == "passes":
            for _ in range(state["steps"]):
                _passes(sim, state["dt"])
        else:
            if state["drive"] == "replay":
                sim.replay()
            else:
                sim.step_many(state["steps"])
            sim.sync()
        p, u, flags = sim.get_state()
        return {"p": p, "u": u, "flags": flags, "counters": sim.counters()}
    if state["kind"] == "batch":
        state["batch"].solve()
        uu, pp, result, counts = state["batch"].get()
        return {"uu": uu, "pp": pp, "result": result, "counts": list(counts)}
    rc = hip.lib().kz_implicit_solve_noalloc(
        state["n"], state["pp_in"].data_ptr(), state["geom"].data_ptr(), state["dt"].data_ptr(),
        state["uu"].data_ptr(), state["pp"].data_ptr(), state["result"].data_ptr(), state["counts"].data_ptr(),
        ctypes.byref(state["physics"]), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    if rc:
        raise RuntimeError(T.ERRORS.get(rc, rc))
    return {k: state[k] for k in ("uu", "pp", "result", "counts")}


def work(case):
    """Compulsory bytes and counted FP64 operations.

    A step reads and writes p and u (416 B per zone) and reads the metric (29
    doubles, the symmetric halves of g and all of G with three scalars, at the
    centre and at one face per active dimension) and 40 Christoffels; the
    state is written out once a pass.  Operations are
    those of its two implicit solves, 28 135 each on the 384x360 torus; the
    passes' driver does one solve per step.  A batch cell takes 134 811
    operations over its ladder."""
    if case["kind"] == "run":
        zones = case["nx"] * case["ny"] * case["nz"]
        dims = 3 if case["nz"] > 1 else 2
        per_step = 4 * 104 + 8 * (29 * (1 + dims) + 40)
        solves = 1 if case["drive"] == "passes" else 2
        return {"bytes": zones * (per_step * case["steps"] + 2 * 104 + 24),
                "flops": zones * solves * 28135.0 * case["steps"]}
    n = case["cells"]
    return {"bytes": n * (8.0 * (T.NV + 30 + 1) + 8.0 * 2 * T.NV + 24), "flops": n * 134811.0}


def exact(case, seed):
    return None
