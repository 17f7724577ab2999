"""The end of an iteration with fewer workgroups per section (batches of more than 8
and of 48 instances or more), sections of more parts than workgroups, against the
same passages alone: the same parts added in the same order, so the same bits."""
import numpy as np
import pytest

from fv3d import cases
from fv3d.solver import GpuSolver

pytestmark = pytest.mark.gpu


def passages(n, ni, nj):
    cs = [cases.annular_passage(ni=ni, nj=nj, nk_blocks=(5, 6, 4), max_iter=6, seed=q, rpm=3000.0) for q in range(n)]
    for q, c in enumerate(cs):
        c.cfg.p_out *= 1.0 + 0.001 * q
    return cs


# sections of 2,300 cells (nine parts), 20 cells (one part) and 8,256 cells (33: every part, one of two rounds)
@pytest.mark.parametrize("n,ni,nj", [(8, 50, 46), (9, 50, 46), (47, 50, 46), (48, 50, 46), (48, 5, 4), (9, 96, 86)])
def test_history_equals_lone(n, ni, nj):
    print(f"case {n} instances, section {ni} x {nj}", flush=True)
    cs = passages(n, ni, nj)
    g = GpuSolver(cs)
    h = g.iterate(3)
    hg = g.iterate(5, graph=True)
    for q in (0, n // 2, n - 1):
        a = GpuSolver(cs[q])
        np.testing.assert_array_equal(a.iterate(3), h[:, q, :])
        np.testing.assert_array_equal(a.iterate(5, graph=True), hg[:, q, :])
        a.close()
    g.close()
