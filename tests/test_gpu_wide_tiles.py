"""The residual kernels' wide workgroups on small grids: tile counts at both
sides of the rules (256 for the viscous kernel, 512 for the convective one) and
ragged tiles, every reconstruction, against tiles of another shape, which run
256 threads: the same faces and sums, so the same bits."""
import numpy as np
import pytest

from fv3d import cases
from fv3d.solver import GpuSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("var", [200, 100, 300])
@pytest.mark.parametrize("shape", [(3, 3, 3), (9, 7, 33), (16, 64, 64), (17, 64, 64), (32, 64, 64), (33, 64, 64)])
def test_residual(shape, var):
    ni, nj, nk = shape
    print(f"case wide tiles {shape} variables {var}", flush=True)
    out = []
    for tiles in ((0, 0, 0), (2, 2, 2)):
        g = GpuSolver(cases.bump_channel(ni=ni, nj=nj, nk=nk, seed=ni, viscous=True, len_ref=1e-3, recon_var=var,
                                         max_iter=2))
        g.set_tiles(tiles)
        g.call("lusgs")
        out.append((g.get(1, "res"), g.get(1, "cv")))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
