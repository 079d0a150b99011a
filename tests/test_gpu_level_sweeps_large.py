"""Full steps on 2-D multicolour numberings whose levels are at and over the
131,072 cells up to which a level is split by face entries (beyond, one thread
per cell), against the oracle, bit for bit: every viscous model, SA, and
increments that need SolutionFix (raised by that form of the sweeps too)."""
import numpy as np
import pytest

from oneflow_amd import meshgen
from tests.test_gpu_level_sweeps import begin, start

pytestmark = pytest.mark.gpu

GRIDS = {  # two levels each, of half the cells
    "quads_131072": lambda: meshgen.box2d(512, 512, jitter=0.2, seed=1),
    "quads_131080": lambda: meshgen.box2d(1808, 145, x1=12.0, jitter=0.2, seed=2),
    "tris_140000": lambda: meshgen.box2d(400, 350, tri=True, jitter=0.2, seed=3),
}


@pytest.mark.parametrize("grid", list(GRIDS))
def test_large_levels_bitwise(grid):
    from oneflow_amd.solver import Solver
    g = GRIDS[grid]()
    g = meshgen.renumber(g, meshgen.multicolor_order(g))
    for opt in ("sa", "euler", "laminar_sr1", "fix"):
        cfg, ora, q, t = start(g, opt)
        gpu = Solver(g, cfg)
        print(f"[large levels] {grid} {opt} cells={g.n_cells} levels={gpu.n_levels}", flush=True)
        assert gpu.n_levels == 2 and g.n_cells == 2 * int(grid.split("_")[1])
        for s in (gpu, ora):
            begin(s, q, t)
            s.iterate(5, 1 if opt == "fix" else 2)
        C = g.n_cells
        for n in ("DQ", "Q") + (("TURBDQ", "TURBQ", "VIST") if opt == "sa" else ()):
            a, b = gpu.get(n)[..., :C], ora.get(n)[..., :C]
            assert np.isfinite(b).all() and np.array_equal(a, b), (opt, n, float(np.max(np.abs(a - b))))
        gpu.close()
