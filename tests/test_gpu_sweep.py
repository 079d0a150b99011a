"""The pipelined LU-SGS sweeps (numberings with many narrow dependency levels)
against the oracle, bit for bit, at the shapes where they can go wrong: one
range and many, levels narrower and wider than the cells a wave takes, every
dependency count, halos, 3-D cells, Euler and viscous, both SA and NS."""
import numpy as np
import pytest

from oneflow_amd import meshgen
from oneflow_amd.config import CaseConfig
from oracle.pyoracle import OracleCase

pytestmark = pytest.mark.gpu


def scrambled(g, block, seed):
    """Cells renumbered: blocks of `block` consecutive cells, each in random order (more dependencies per cell)."""
    rng = np.random.default_rng(seed)
    order = np.concatenate([b + rng.permutation(min(block, g.n_cells - b)) for b in range(0, g.n_cells, block)])
    return meshgen.renumber(g, order)


GRIDS = {
    "chain": lambda: meshgen.box2d(70, 1),                                     # one cell per level, one range
    "strip": lambda: meshgen.box2d(90, 3, jitter=0.2),
    "quads": lambda: meshgen.box2d(61, 53, jitter=0.2),                        # several ranges, wide levels
    "tris": lambda: meshgen.box2d(47, 41, tri=True, jitter=0.1),
    "tris_scrambled": lambda: scrambled(meshgen.box2d(70, 33, tri=True), 60, 2),
    "quads_scrambled": lambda: scrambled(meshgen.box2d(80, 40), 9, 1),
    "hex": lambda: meshgen.box3d(30, 21, 22),
    "tets": lambda: meshgen.box3d(60, 7, 5, kind="tet"),
}


@pytest.mark.parametrize("grid", list(GRIDS))
@pytest.mark.parametrize("opt", ["sa", "euler", "laminar_sr1"])
def test_pipelined_sweeps_bitwise(grid, opt):
    from oneflow_amd.solver import Solver
    g = GRIDS[grid]()
    if opt == "sa":
        g.bc_type[: max(1, g.n_bfaces // 5)] = 2  # walls for the wall distance
    kw = dict(sa=dict(vismodel=3), euler=dict(vismodel=0), laminar_sr1=dict(vismodel=1, visSRModel=1))[opt]
    cfg = CaseConfig(dim=g.dim, ischeme=1, ilim=-1, mach_ref=0.5, aoa_degree=2.0, reynolds=1e4, **kw)
    gpu, ora = Solver(g, cfg), OracleCase(g, cfg)
    print(f"[sweep] {grid} {opt} cells={g.n_cells} levels={gpu.n_levels}", flush=True)
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
        s.iterate(5, 3)
    C = g.n_cells
    for n in ("DQ", "Q") + (("TURBDQ", "TURBQ") if opt == "sa" else ()):
        a, b = gpu.get(n)[..., :C], ora.get(n)[..., :C]
        assert np.isfinite(b).all() and np.array_equal(a, b), (n, float(np.max(np.abs(a - b))))
    gpu.close()
