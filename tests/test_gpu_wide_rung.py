"""The implicit pass from the size at which the first rung is launched at two
waves per SIMD (768 cells per CU: 196 608 on 256 CUs), in every variant that a
caller can get: one grid and a run group whose cells add up to exactly that
size, without and with the synchrotron bridge, in the launch the size selects
and in the persistent launches, whose lanes each take several cells here.  States
of the independent-cell batch are planted in every run, so that some cells
need a later rung and some fail the whole ladder.  One CFL step of each equals
the oracle's bit for bit."""
import functools

import pytest
import torch

import kzo
from test_gpu_fullsize import SEED, _threads
from test_gpu_step import assert_same
from koral_zig_amd import abi_types as T
from koral_zig_amd import hip, host, workloads

pytestmark = pytest.mark.gpu
GRIDS = {"grid": ((512, 384, 0.0),), "group": ((384, 256, 0.5), (256, 384, 0.9375))}


@functools.lru_cache(maxsize=3)
def torus(nx, ny, a):
    grid = T.grid_puffy(nx, ny, rmin=T.rmin_for_spin(a))
    ph = T.physics_puffy(bh_spin=a)
    tab = host.metric_tables(grid, dict(host.MP_PUFFY, a=a))
    return grid, tab, host.puffy_prepinit(grid, tab, ph, host.PUFFY_INIT)


def plant(p, grid, seed, n=300):
    """n batch states in interior cells of the padded primitives, no two next
    to each other."""
    ph = T.physics_puffy()
    pp, _, _ = workloads.implicit_batch_inputs(n, seed, ph, lambda q, g: kzo.opac_entry(q, g, ph.gam, ph.opac)[:, 3])
    _, (ngz, ngy, ngx) = T.padded_shape(grid)
    p, per_row = p.copy(), (grid.nx - 16) // 8
    for k in range(n):
        p[ngz, ngy + 16 + 8 * (k // per_row), ngx + 8 + 8 * (k % per_row)] = pp[k]
    return p


def start(make, grid, ph, tab, p0, seed):
    s = make(grid, ph, tab)
    host.init_puffy(s, grid, tab, ph, seed=SEED, p0=p0)
    s.set_state(p=plant(s.get_state()[0], grid, seed))
    s.p2u_domain()
    return s


@functools.lru_cache(maxsize=1)
def oracle(cells, bridge):
    """[(grid, physics, tables, torus, seed, the oracle's run after a step)]"""
    _threads()
    out = []
    for k, run in enumerate(GRIDS[cells]):
        grid, tab, p0 = torus(*run)
        ph = T.physics_puffy(bh_spin=run[2])
        ph.opac.synchrotron_bridge = bridge
        cpu = start(kzo.Sim, grid, ph, tab, p0, 17 + k)
        cpu.step()
        assert cpu.counters()["n_radimp_failures"] > 0
        out.append((grid, ph, tab, p0, 17 + k, cpu))
        print(f"{run} bridge {bridge}: the oracle has stepped", flush=True)
    return out


@pytest.mark.timeout(300)
@pytest.mark.parametrize("cells,bridge,mode", [(c, b, m) for c in GRIDS for b in (0, 1) for m in (0, 2)])
def test_wide_first_rung(cells, bridge, mode):
    size = sum(nx * ny for nx, ny, _ in GRIDS[cells])
    assert size == 196608 and size >= 768 * torch.cuda.get_device_properties(0).multi_processor_count
    runs = oracle(cells, bridge)
    gpus = [start(hip.Sim, *run[:5]) for run in runs]
    if cells == "grid":
        gpus[0].set_implicit_launch(mode)
        gpus[0].step()
    else:
        grp = hip.Group(gpus)
        grp.set_implicit_launch(mode)
        grp.step_many(1)
        grp.sync()
        grp.close()
    for run, gpu in zip(runs, gpus):
        assert_same(run[5], gpu, f"{cells}, bridge {bridge}, launch {mode}")
        gpu.close()
