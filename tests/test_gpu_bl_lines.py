"""Baldwin-Lomax over line lengths at the edges of its forms (groups per line and
cells per thread), against the CPU oracle.  Tolerance as in
test_gpu_viscous.py: the device pow and exp round differently from libm's,
1e-12 of the field's magnitude for one evaluation."""
import numpy as np
import pytest

from fv3d import cases
from fv3d.solver import GpuSolver
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni", [3, 15, 16, 17, 32, 33, 64, 65, 128, 129, 256, 257])
def test_line_lengths(ni):
    case = cases.with_wall_shear(cases.bump_channel(ni=ni, nj=5, nk=9, seed=200 + ni, viscous=True, len_ref=1e-3,
                                                    max_iter=2))
    case.cfg.turbulence = 100
    print(f"case BL lines of {ni} cells", flush=True)
    o, g = O.Oracle(case), GpuSolver(case)
    o.call("lusgs")
    g.call("lusgs")
    a, b = g.get(1, "mut"), o.get(1, "mut")
    assert np.max(np.abs(b)) > 0.0
    assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b))
