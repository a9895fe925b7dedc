"""The flat collide-stream form (rows that are no whole chunks of 256 nodes) where its
workgroups end: layers of one node less than, exactly and one more than whole
workgroups, rows shorter and longer than a workgroup, the smallest lattice, each gratio
and both drivings, against the oracle: bit for bit under a constant force, 1e-12 of the
largest value under the flux controller (its sum is taken in another order)."""
import numpy as np
import pytest

from helpers import Oracle, dnsg, relmax

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 1), (17, 15, 1), (16, 16, 1), (257, 3, 1), (8, 4, 2), (51, 5, 3), (171, 2, 3), (33, 7, 4), (300, 2, 1)]


@pytest.mark.parametrize("force", ["const", "flux"])
@pytest.mark.parametrize("x,y,gr", SHAPES)
def test_flat_edges(x, y, gr, force):
    p = dnsg.make_params(xdv=x, ydv=y, zdv=8, gratio=gr, zds=6, tau_c=0.53, ub=0.05, force_mode=force, g_const=2e-5,
                         CFL=1.0, pattern="pslip", gxplussize=gr * x - 1, wxplussize=1, gyplussize=1,
                         wyplussize=gr * y - 1, init_kind="laminar_noise", seed=9, u_max=0.05, noise=0.1)
    o, s = Oracle(p), dnsg.Solver(p)
    o.init_seeded()
    s.init_state()
    do, ds = o.run(4), s.step(4)
    a, b = s.download(), o.state()
    s.close()
    for k in ("coarse", "lower", "upper", "lin", "uin"):
        if force == "const":
            assert np.array_equal(a[k], b[k]), k
        else:
            assert relmax(a[k], b[k]) <= 1e-12, k
    for f in ("momentum", "density", "str_up", "str_down"):
        assert np.allclose(ds[f], do[f], rtol=1e-10, atol=1e-16), f
