"""The viscous residual's two workgroup sizes (768 threads up to 256 tiles, 256
beyond) against each other, on grids that two tile shapes cut into counts on
either side of the rule, and the smaller workgroups against the CPU oracle.  Tolerance of the
latter as in test_gpu_viscous.py: 1e-12 of the field's magnitude for one iteration."""
import numpy as np
import pytest

from fv3d import cases
from fv3d.solver import GpuSolver
import oracle as O

pytestmark = pytest.mark.gpu

WIDE = 256   # kWideVisc of csrc/fv3d_kernels.h
SHAPE = {0: (4, 4, 16), 2: (4, 8, 8), 4: (8, 8, 4)}


def tiles(cells, shape):
    """Tiles of a one-block grid, padded to whole rounds over the eight XCDs."""
    n = 1
    for c, t in zip(cells, SHAPE[shape]):
        n *= -(-c // t)
    return -(-n // 8) * 8


@pytest.mark.parametrize("cells,few,many", [((64, 68, 8), 2, 0), ((63, 67, 7), 2, 0), ((4, 4, 1040), 0, 4),
                                            ((3, 4, 1043), 0, 4)])
def test_same_bits(cells, few, many):
    print(f"case {cells}: {tiles(cells, few)} and {tiles(cells, many)} tiles", flush=True)
    assert tiles(cells, few) <= WIDE < tiles(cells, many)
    out = []
    for shape in (few, many):
        g = GpuSolver(cases.bump_channel(ni=cells[0], nj=cells[1], nk=cells[2], seed=cells[1], viscous=True,
                                         len_ref=1e-3, max_iter=2))
        g.set_tiles((shape, shape, shape))
        g.call("lusgs")
        out.append((g.get(1, "res"), g.get(1, "dq"), g.get(1, "cv")))
        g.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("cells,shape", [((34, 66, 50), 0), ((64, 68, 8), 0), ((3, 4, 1043), 4), ((4, 4, 1040), 0)])
def test_oracle(cells, shape):
    print(f"case {cells}, shape {shape}: {tiles(cells, shape)} tiles against the oracle", flush=True)
    c = cases.bump_channel(ni=cells[0], nj=cells[1], nk=cells[2], seed=7, viscous=True, len_ref=1e-3, max_iter=2)
    o = O.Oracle(c)
    o.call("lusgs")
    g = GpuSolver(c)
    g.set_tiles((0, shape, 0))
    g.call("lusgs")
    for f in ("res", "dq", "cv"):
        a, r = g.get(1, f), o.get(1, f)
        assert np.max(np.abs(a - r)) <= 1e-12 * max(np.max(np.abs(r)), 1e-300), f
    g.close()
