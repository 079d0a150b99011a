"""Waits of the pipelined LU-SGS sweeps that give up (the guard's limit set to
almost nothing from the host): every kernel ends, and an increment is either
the oracle's bits or NaN, never another number.  With the limit back at the
schedule's, the same context sweeps as before."""
import numpy as np
import pytest

from oneflow_amd import meshgen
from oneflow_amd.config import CaseConfig
from oracle.pyoracle import OracleCase

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("polls", [1, 100, 400, 2000])
@pytest.mark.parametrize("grid", ["strip", "quads", "hex"])
def test_given_up_waits(grid, polls):
    from oneflow_amd.solver import Solver
    g = {"strip": lambda: meshgen.box2d(90, 3, jitter=0.2), "quads": lambda: meshgen.box2d(90, 71, jitter=0.2),
         "hex": lambda: meshgen.box3d(30, 21, 22)}[grid]()
    g.bc_type[: g.n_bfaces // 5] = 2  # walls for the wall distance
    cfg = CaseConfig(dim=g.dim, ischeme=1, ilim=-1, vismodel=3, mach_ref=0.5, aoa_degree=2.0, reynolds=1e4)
    gpu, ora = Solver(g, cfg), OracleCase(g, cfg)
    print(f"[sweep guard] {grid} polls={polls} cells={g.n_cells} levels={gpu.n_levels}", flush=True)
    rng = np.random.default_rng(3)
    for s in (gpu, ora):
        s.init_freestream()
    q, t = ora.get("Q"), ora.get("TURBQ")
    q[:, : g.n_cells] *= 1.0 + 0.02 * rng.standard_normal((5, g.n_cells))
    t[: g.n_cells] *= 1.0 + 0.5 * rng.random(g.n_cells)
    for s in (gpu, ora):
        s.set("Q", q)
        s.set("TURBQ", t)
        s.ns_boundary()
        s.sa_boundary()
        s.timestep(5)
        s.residual_ns()
        s.residual_sa()
    ora.lusgs_ns()
    ora.lusgs_sa()
    for limit in (polls, 0):
        gpu._check(gpu._L.ofx_set_sweep_polls(gpu.h, limit))
        gpu.lusgs_ns()
        gpu.lusgs_sa()
        gpu.sync()
        for n in ("DQ", "TURBDQ"):
            a, b = gpu.get(n)[..., : g.n_cells], ora.get(n)[..., : g.n_cells]
            lost = np.isnan(a)
            print(f"[sweep guard]   limit {limit} {n}: {int(lost.sum())} of {a.size} NaN", flush=True)
            assert np.isfinite(b).all() and np.array_equal(a[~lost], b[~lost])
            assert limit or not lost.any()
            if limit == 1:
                assert lost.any()
    gpu.close()
