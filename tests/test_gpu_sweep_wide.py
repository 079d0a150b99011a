"""The pipelined sweeps' wide ranges (long fronts of many cells: at least 128
cells a level and as many levels) against the oracle, bit for bit."""
import numpy as np
import pytest

from oneflow_amd import meshgen
from oneflow_amd.config import CaseConfig
from oracle.pyoracle import OracleCase

pytestmark = pytest.mark.gpu

GRIDS = {
    "tris": lambda: meshgen.box2d(200, 150, tri=True, jitter=0.1),
    "quads": lambda: meshgen.box2d(300, 261, jitter=0.1),
    "quads_narrow": lambda: meshgen.box2d(300, 201, jitter=0.1),  # below the line
}


@pytest.mark.parametrize("grid", list(GRIDS))
def test_wide_ranges_bitwise(grid):
    from oneflow_amd.solver import Solver
    g = GRIDS[grid]()
    g.bc_type[: g.n_bfaces // 5] = 2  # walls for the wall distance
    cfg = CaseConfig(dim=2, ischeme=1, ilim=-1, vismodel=3, mach_ref=0.5, aoa_degree=2.0, reynolds=1e4)
    gpu, ora = Solver(g, cfg), OracleCase(g, cfg)
    per = g.n_cells // gpu.n_levels
    print(f"[wide sweeps] {grid} cells={g.n_cells} levels={gpu.n_levels}", flush=True)
    assert (per >= 128 and gpu.n_levels >= per) == (grid != "quads_narrow")
    rng = np.random.default_rng(5)
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
        s.iterate(5, 2)
    for n in ("DQ", "Q", "TURBDQ", "TURBQ"):
        a, b = gpu.get(n)[..., : g.n_cells], ora.get(n)[..., : g.n_cells]
        assert np.isfinite(b).all() and np.array_equal(a, b), n
    gpu.close()
