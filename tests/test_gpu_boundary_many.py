"""Ghost fills and exchange of a batch with many transfers (two launches, the layers
of a K face apart) against the same passages alone (one launch, layers together): the
same transfers, so the same bits."""
import numpy as np
import pytest

from fv3d import cases
from fv3d.solver import GpuSolver

pytestmark = pytest.mark.gpu

MANY = 1500000   # kManyExch of csrc/fv3d_ctx.hip


def transfers(c):
    """Both directions and both layers of every two-sided patch."""
    return sum(4 * int(np.prod([p.rng[2 * e + 1] - p.rng[2 * e] + 1 for e in range(3)]))
               for p in c.patches if p.kind in ("interior", "periodic"))


@pytest.mark.parametrize("n", [140, 180])
def test_batch_equals_lone(n):
    cs = cases.passage_batch(n=n, seed=3, min_cells=1.5e4, max_cells=6e4, design_rpm=0.0, max_iter=10)
    total = sum(transfers(c) for c in cs)
    print(f"case {n} passages, {total:,} transfers", flush=True)
    assert (total > MANY) == (n == 180)
    g = GpuSolver(cs, precision=1)
    h = g.iterate(3, graph=True)
    for q in (0, n // 2, n - 1):
        assert transfers(cs[q]) < MANY
        a = GpuSolver(cs[q], precision=1)
        np.testing.assert_array_equal(a.iterate(3, graph=True), h[:, q, :])
        for b in range(1, len(cs[q].blocks) + 1):
            for f in ("cv", "dKS_cv", "dKP_pv", "dJS_cv"):
                np.testing.assert_array_equal(a.get(b, f), g.get(b, f, inst=q + 1))
        a.close()
    g.close()
