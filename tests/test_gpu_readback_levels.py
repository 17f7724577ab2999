"""Fields of two grid levels read in turn through the context's one staging buffer
(fine fields from one chunk and from two), against a context that reads one of
them only: the same values, whatever was read before."""
import numpy as np
import pytest

from fv3d import cases
from fv3d.solver import GpuSolver

pytestmark = pytest.mark.gpu


def solver(n):
    c = cases.bump_channel(ni=n, nj=n, nk=n, seed=n, max_iter=10)
    c.cfg.use_multigrid, c.cfg.reuse_solution, c.cfg.initial, c.cfg.coarse_iter = "Y", "N", "U", 2
    g = GpuSolver(c)
    g.iterate(4)
    return g


@pytest.mark.parametrize("n", [6, 32, 72])
def test_levels_in_turn(n):
    print(f"case levels in turn {n}^3", flush=True)
    g = solver(n)
    seen = [(f, level, g.get(1, f, level=level)) for f in ("cv", "res", "pv") for level in (1, 2, 1)]
    g.close()
    for f, level, v in seen:
        a = solver(n)
        np.testing.assert_array_equal(a.get(1, f, level=level), v, err_msg=f"{f}, level {level}")
        a.close()
