"""The backward sweep's planes into the cell box, at plane counts around the steps
a plane is spread over and at blocks that end inside a tile: dQ and dnu~ have
the bits of the per-hyperplane form (the reference's schedule).  The FP32
operator, which has no such form, against the FP64 one: its dQ differs by the
rounding of its products, some hundred of them in a chain, so 1e-3 of the
largest value holds where a misplaced cell is off by that value itself."""
import numpy as np
import pytest

from fv3d import cases
from fv3d.solver import GpuSolver

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3, 3), (18, 4, 16), (19, 5, 17), (20, 3, 15), (21, 8, 33), (41, 6, 48)]


def build(ni, nj, nk):
    return cases.with_sa(cases.annular_passage(ni=ni, nj=nj, nk_blocks=(nk, 5), viscous=True, len_ref=1e-3, seed=ni))


@pytest.mark.parametrize("shape", SHAPES)
def test_planes(shape):
    print(f"case sweep store {shape}", flush=True)
    a, b = GpuSolver(build(*shape)), GpuSolver(build(*shape), debug=2)
    np.testing.assert_array_equal(a.iterate(2), b.iterate(2))
    for blk in (1, 2):
        for f in ("dq", "dev", "cv", "ev"):
            np.testing.assert_array_equal(a.get(blk, f), b.get(blk, f))


@pytest.mark.parametrize("shape", SHAPES)
def test_fp32_operator(shape):
    print(f"case sweep store FP32 {shape}", flush=True)
    a, b = GpuSolver(build(*shape)), GpuSolver(build(*shape), precision=1)
    for g in (a, b):
        g.call("lusgs")
    for blk in (1, 2):
        for f in ("dq", "dev"):
            x, y = a.get(blk, f), b.get(blk, f)
            x, y = x.reshape(x.shape[0], x.shape[1], x.shape[2], -1), y.reshape(x.shape[0], x.shape[1], x.shape[2], -1)
            for c in range(x.shape[-1]):
                s = np.max(np.abs(x[..., c]))
                assert np.max(np.abs(x[..., c] - y[..., c])) <= 1e-3 * s, f"block {blk} {f} component {c}"
