"""Ghost fills and transfers in one launch, and in two where a boundary patch and
a transfer fill the same cells (the transfer is the later one, as in the
reference's order of patches), against the CPU oracle.  Tolerance as in
test_gpu_passage.py."""
import numpy as np
import pytest

from fv3d import cases
from fv3d.refio import Patch
from fv3d.solver import GpuSolver
import oracle as O

pytestmark = pytest.mark.gpu

FIELDS = ("dIS_cv", "dIP_cv", "dJS_cv", "dJP_cv", "dKS_cv", "dKP_cv", "dJS_pv", "dKP_pv", "res", "dq", "cv", "pv")
EXTRA = {"none": None, "wall over an interior patch": Patch("wall", 2, 6, (2, 4, 3, 6, 7, 7)),
         "wall over a periodic patch": Patch("wall", 2, 4, (2, 4, 9, 9, 2, 5))}


@pytest.mark.parametrize("extra", list(EXTRA))
def test_order(extra):
    c = cases.annular_passage(ni=6, nj=8, nk_blocks=(5, 6, 4), max_iter=6, seed=70, rpm=5000.0)
    if EXTRA[extra]:
        c.patches.append(EXTRA[extra])
    print(f"case boundary order, {extra}", flush=True)
    o, g = O.Oracle(c), GpuSolver(c)
    o.call("lusgs")
    g.call("lusgs")
    for b in range(1, 4):
        for f in FIELDS:
            a, r = g.get(b, f), o.get(b, f)
            assert np.max(np.abs(a - r)) <= 1e-12 * max(np.max(np.abs(r)), 1e-300), f"block {b} {f}"
