"""The budget with 1, 2, 4 and 8 rows a thread (grids of a few thousand nodes to two
million), the number of rows no multiple of that, rows that start anywhere in a workgroup:
every profile against the oracle on the same snapshot, 1e-10 of its scale."""
import numpy as np
import pytest

from helpers import budget_scales, dnsg, oracle_budget

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x,y,z,zds,gr,prec", [(31, 23, 14, 8, 2, "fp64"), (97, 63, 40, 9, 2, "fp16"),
                                               (143, 71, 48, 10, 2, "fp64"), (199, 107, 106, 8, 1, "fp32")])
def test_profiles(x, y, z, zds, gr, prec):
    p = dnsg.make_params(xdv=x, ydv=y, zdv=z, gratio=gr, zds=zds, Rebs=40.0, ub=0.03, CFL=1.0, force_mode="const",
                         g_const=2e-5, precision=prec, init_kind="laminar_noise", seed=3, u_max=0.05, noise=0.2)
    s = dnsg.Solver(p)
    s.init_state()
    s.step(5)
    got = s.budget2d()
    ref = oracle_budget(p, {g: s.velocity(g) for g in range(3)})
    s.close()
    for kind, a, b in zip(("turb", "vort", "ke"), got, ref):
        assert np.all(np.abs(a - b) <= 1e-10 * budget_scales(kind, b)[:, None] + 1e-300), kind
