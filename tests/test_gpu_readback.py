"""Fields read back cell by cell, from one staging chunk and from two (a field
beyond 16 MiB): the uploaded start state must come back value for value, and
the box arrays must agree with the interior ones where both exist."""
import numpy as np
import pytest

from fv3d import cases
from fv3d.solver import GpuSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj,nk", [(5, 3, 7), (33, 18, 41), (72, 68, 69)])
def test_state_comes_back(ni, nj, nk):
    print(f"case read-back {ni}x{nj}x{nk}", flush=True)
    case = cases.with_sa(cases.with_wall_shear(cases.bump_channel(ni=ni, nj=nj, nk=nk, seed=nk, viscous=True, len_ref=1e-3)))
    st = case.states[0]
    g = GpuSolver(case)
    pv, cv, ev = g.get(1, "pv"), g.get(1, "cv"), g.get(1, "ev")
    inner = (slice(1, -1),) * 3
    for q, name in enumerate(("rho", "u", "v", "w", "p", "T")):
        np.testing.assert_array_equal(pv[inner + (q,)], st[name])
    np.testing.assert_array_equal(cv[inner + (0,)], st["rho"])
    np.testing.assert_array_equal(cv[inner + (4,)], st["rhoE"])
    np.testing.assert_array_equal(ev[inner], st["nut"])
    # an interior array against the box array of the same quantity: dQ = Q' - Q
    # of one LU-SGS step (Q of order one: within two roundings of the sum)
    g.call("lusgs")
    dq, cv1 = g.get(1, "dq"), g.get(1, "cv")
    assert np.max(np.abs(cv1[inner] - cv[inner] - dq)) <= 4 * np.finfo(float).eps * np.max(np.abs(cv))
    assert g.get(1, "vol").shape == (ni, nj, nk) and np.all(g.get(1, "vol") > 0)
    g.close()
