"""Replayed iterations in groups: counts below, at and past the iterations one
graph holds, from the coarse start-up phase and from the middle of a run, give
the eager run's bits."""
import numpy as np
import pytest

from fv3d import cases
from fv3d.solver import GpuSolver

pytestmark = pytest.mark.gpu


def build(name):
    if name == "flipped passage":
        return cases.annular_passage(ni=6, nj=8, nk_blocks=(5, 6, 4), max_iter=30, seed=75, rpm=5000.0,
                                     periodic_from_high=True)
    c = cases.bump_channel(ni=8, nj=8, nk=16, seed=51, max_iter=30)
    if name == "two-grid bump":
        c.cfg.use_multigrid, c.cfg.reuse_solution = "Y", "N"
        c.cfg.coarse_iter, c.cfg.initial, c.cfg.outlet_angle = 3, "U", (0.0, 0.0, 1.0)
    return c


@pytest.mark.parametrize("name", ["bump", "flipped passage", "two-grid bump"])
@pytest.mark.parametrize("counts", [(3, 4), (5, 8), (7, 1, 4, 2), (9,)])
def test_grouped_replay(name, counts):
    print(f"case {name} counts {counts}", flush=True)
    a, b = GpuSolver(build(name)), GpuSolver(build(name))
    ha = a.iterate(sum(counts))
    hb = np.concatenate([b.iterate(n, graph=True) for n in counts])
    np.testing.assert_array_equal(ha, hb)
    for blk in range(1, len(build(name).blocks) + 1):
        np.testing.assert_array_equal(a.get(blk, "cv"), b.get(blk, "cv"))
