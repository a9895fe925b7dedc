"""The interface fill's two forms (substeps before the last, which read three plane levels,
and the last, which reads the newest) and the sharing of the directions over workgroups,
against the oracle bit for bit in FP64 under a constant force: lattices of less than one
32 x 8 tile, of exactly one, ragged against it, and of tiles enough that a workgroup takes
several units of directions."""
import numpy as np
import pytest

from helpers import Oracle, dnsg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x,y,gr", [(6, 2, 2), (32, 8, 2), (33, 9, 1), (31, 17, 2), (65, 15, 3), (36, 12, 4), (256, 96, 2)])
def test_fill_matches_oracle(x, y, gr):
    p = dnsg.make_params(xdv=x, ydv=y, zdv=9, gratio=gr, zds=6, tau_c=0.53, ub=0.05, force_mode="const", g_const=2e-5,
                         CFL=1.0, precision="fp64", init_kind="laminar_noise", seed=7, u_max=0.05, noise=0.1)
    o = Oracle(p, threads=4)
    s = dnsg.Solver(p)
    s.init_state()
    o.init_seeded()
    o.run(3)
    s.step(3)
    g, ref = s.download(), o.state()
    for k in ("coarse", "lower", "upper", "lin", "uin"):
        assert np.array_equal(g[k], ref[k]), k
