"""The interface fill with 2, 3, 5, 7 and 19 workgroups a tile (on a device of 256 CUs;
10, 1 and 19 in FP64 are met by the other sizes).  FP64 against the oracle bit for bit.
FP32 and FP16 planes after one step, against the oracle's FP64 step from the same start:
rounding of shifted values of at most 0.05 leaves 1e-6 and, in FP16 storage, 1e-4 of
room many times over, where a value of another direction, or one not written, is off by
more than 1e-3."""
import numpy as np
import pytest

from helpers import Oracle, dnsg

pytestmark = pytest.mark.gpu


def both(x, y, gr, prec, n):
    kw = dict(xdv=x, ydv=y, zdv=8, gratio=gr, zds=max(5, gr + 3), tau_c=0.53, ub=0.05, force_mode="const", g_const=2e-5,
              CFL=1.0, init_kind="laminar_noise", seed=7, u_max=0.05, noise=0.1)
    o, s = Oracle(dnsg.make_params(**kw), threads=8), dnsg.Solver(dnsg.make_params(precision=prec, **kw))
    o.init_seeded(), s.init_state()
    o.run(n), s.step(n)
    out = s.download(), o.state()
    s.close(), o.close()
    return out


# tiles of both bands: 64 at gratio 4 (7), 90 (5), 160 and 256 at gratio 2 (3 or 5), 256 at gratio 3 (2)
@pytest.mark.parametrize("x,y,gr", [(100, 60, 4), (143, 71, 2), (250, 80, 2), (256, 128, 2), (256, 128, 3)])
def test_fp64(x, y, gr):
    g, ref = both(x, y, gr, "fp64", 2)
    for k in ("coarse", "lower", "upper", "lin", "uin"):
        assert np.array_equal(g[k], ref[k]), k


# 16 and 30 tiles (19), 96 (5)
@pytest.mark.parametrize("prec", ["fp32", "fp16"])
@pytest.mark.parametrize("x,y,gr", [(48, 30, 4), (80, 37, 3), (190, 60, 4)])
def test_shifted(x, y, gr, prec):
    g, ref = both(x, y, gr, prec, 1)
    for k in ("coarse", "lower", "upper"):
        assert np.max(np.abs(g[k] - ref[k])) <= {"fp32": 1e-6, "fp16": 1e-4}[prec], k
