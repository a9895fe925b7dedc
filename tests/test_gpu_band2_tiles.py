"""The two-substep band kernel at the edges of its tiles (62 columns in FP64, 124 in FP32
and FP16, by 10 rows) against one collide-stream launch per substep, bit for bit under a
constant force: lattices one tile wide, exactly two, one column or row more and less,
rows shorter than a tile, the periodic edge inside and between tiles, thin and deep
bands.  Both paths run the same collisions on the same values, so no tolerance."""
import numpy as np
import pytest

from helpers import dnsg

pytestmark = pytest.mark.gpu

# coarse (x, y), fluid layers per band, pattern; the bands have 2x by 2y columns
SHAPES = [(31, 5, 4, "none"), (62, 10, 5, "pslip"), (63, 11, 4, "rslip"), (61, 4, 7, "sslip"), (124, 6, 4, "pslip"),
          (125, 21, 4, "none"), (6, 2, 16, "rslip")]


@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16"])
@pytest.mark.parametrize("x,y,zds,pattern", SHAPES)
def test_tile_edges(x, y, zds, pattern, prec, monkeypatch):
    kw = dict(xdv=x, ydv=y, zdv=9, gratio=2, zds=zds, tau_c=0.53, ub=0.05, force_mode="const", g_const=2e-5, CFL=1.0,
              precision=prec, pattern=pattern, gxplussize=1, wxplussize=1, gyplussize=1, wyplussize=1,
              init_kind="laminar_noise", seed=5, u_max=0.05, noise=0.1)
    got = []
    for band2 in "10":
        monkeypatch.setenv("DNSG_BAND2", band2)
        s = dnsg.Solver(dnsg.make_params(**kw))
        assert s.band_launch_substeps() == 1 + int(band2)
        s.init_state()
        rec = s.step(5)
        got.append((s.download(), rec))
        s.close()
    (a, ra), (b, rb) = got
    for k in ("coarse", "lower", "upper", "lin", "uin"):
        assert np.array_equal(a[k], b[k]), k
    for f in ("momentum", "density", "str_up", "str_down"):  # the same FP64 values summed in another order
        assert np.allclose(ra[f], rb[f], rtol=1e-10, atol=0), f
