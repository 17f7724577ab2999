"""Fields on both sides of the size up to which they are read as one copy of the
cell box (160 KB a component, 512 KB in all): the uploaded start state must come
back value for value, whichever way its fields take."""
import numpy as np
import pytest

from fv3d import cases
from fv3d.solver import GpuSolver

pytestmark = pytest.mark.gpu


# box per component 1, 62, 83 (cv and pv whole), 95 (cv whole, pv not), 108 (ev only), 154 and 171 KB
@pytest.mark.parametrize("ni,nj,nk", [(3, 3, 3), (18, 18, 18), (20, 20, 20), (21, 21, 21), (22, 22, 22), (25, 25, 25),
                                      (26, 26, 26), (3, 5, 600)])
def test_state_comes_back(ni, nj, nk):
    print(f"case small read-back {ni}x{nj}x{nk}, {(ni + 2) * (nj + 2) * (nk + 2) * 8 / 1024:.0f} KB a component", flush=True)
    case = cases.with_sa(cases.with_wall_shear(cases.bump_channel(ni=ni, nj=nj, nk=nk, seed=nk, viscous=True, len_ref=1e-3)))
    st = case.states[0]
    g = GpuSolver(case)
    inner = (slice(1, -1),) * 3
    pv, cv = g.get(1, "pv")[inner], g.get(1, "cv")[inner]
    for q, name in enumerate(("rho", "u", "v", "w", "p", "T")):
        np.testing.assert_array_equal(pv[..., q], st[name])
    np.testing.assert_array_equal(cv[..., 0], st["rho"])
    np.testing.assert_array_equal(cv[..., 4], st["rhoE"])
    np.testing.assert_array_equal(g.get(1, "ev")[inner], st["nut"])
    # interior arrays: dQ = Q' - Q of one LU-SGS step (Q of order one: within two
    # roundings of the sum), and volumes in place
    g.call("lusgs")
    cv1 = g.get(1, "cv")[inner]
    assert np.max(np.abs(cv1 - cv - g.get(1, "dq"))) <= 4 * np.finfo(float).eps * np.max(np.abs(cv))
    assert np.all(g.get(1, "vol") > 0) and np.all(g.get(1, "dt") > 0)
    g.close()
