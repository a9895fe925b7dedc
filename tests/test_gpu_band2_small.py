"""The two-substep band kernel's small tiles (62 columns by 6 rows, one node per lane, in
FP64 and FP32; DNSG_BAND2=2) at their edges, and both kinds of tile under the flux
controller, against one collide-stream launch per substep (DNSG_BAND2=0).  Under a constant
force the same collisions run on the same values: bit for bit, and sums of the same FP64
values in another order to 1e-10.  Under the flux controller the force feeds back from such
sums: the states agree to the tier's rounding (1e-12 of the largest value in FP64, 1e-5 in
FP32, 1e-2 in FP16 storage).  Lattices one tile wide, exactly two, one column or row more
and less, rows shorter than a tile, thin and deep bands; for the flux controller more
columns and rows than one tile of either kind, ragged, the periodic edge inside a tile."""
import numpy as np
import pytest

from helpers import dnsg, relmax

pytestmark = pytest.mark.gpu
KEYS = ("coarse", "lower", "upper", "lin", "uin")

# coarse (x, y), fluid layers per band, pattern; the bands have 2x by 2y columns
SHAPES = [(31, 3, 4, "none"), (62, 6, 5, "pslip"), (63, 7, 4, "rslip"), (61, 4, 7, "sslip"), (30, 2, 9, "pslip"),
          (94, 13, 4, "none"), (6, 2, 16, "rslip")]


def run(monkeypatch, band2, n, prec, x, y, zds, pattern, force):
    monkeypatch.setenv("DNSG_BAND2", band2)
    s = dnsg.Solver(dnsg.make_params(xdv=x, ydv=y, zdv=9, gratio=2, zds=zds, tau_c=0.53, ub=0.05, force_mode=force,
                                     g_const=2e-5, CFL=1.0, precision=prec, pattern=pattern, gxplussize=1, wxplussize=1,
                                     gyplussize=1, wyplussize=1, init_kind="laminar_noise", seed=5, u_max=0.05, noise=0.1))
    assert s.band_launch_substeps() == (1 if band2 == "0" else 2)
    s.init_state()
    rec = s.step(n)
    st = s.download()
    s.close()
    return st, rec


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("x,y,zds,pattern", SHAPES)
def test_small_tile_edges(x, y, zds, pattern, prec, monkeypatch):
    (a, ra), (b, rb) = (run(monkeypatch, v, 5, prec, x, y, zds, pattern, "const") for v in "20")
    for k in KEYS:
        assert np.array_equal(a[k], b[k]), k
    for f in ("momentum", "density", "str_up", "str_down"):
        assert np.allclose(ra[f], rb[f], rtol=1e-10, atol=0), f


@pytest.mark.parametrize("prec,tile", [("fp64", "1"), ("fp64", "2"), ("fp32", "1"), ("fp32", "2"), ("fp16", "1")])
@pytest.mark.parametrize("x,y", [(97, 11), (62, 13)])
def test_flux_control_over_several_tiles(x, y, prec, tile, monkeypatch):
    (a, ra), (b, rb) = (run(monkeypatch, v, 20, prec, x, y, 5, "pslip", "flux") for v in (tile, "0"))
    tol = {"fp64": 1e-12, "fp32": 1e-5, "fp16": 1e-2}[prec]
    for k in ("coarse", "lower", "upper"):
        assert relmax(a[k], b[k]) <= tol, k
    for f in ("momentum", "density", "flowrate"):
        assert relmax(ra[f], rb[f]) <= tol, f
    assert np.max(np.abs(ra["force"] - rb["force"])) <= tol * 0.05


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("force", ["const", "flux"])
def test_nan_stops_every_path_at_the_same_step(force, prec, monkeypatch):
    """a NaN planted in the middle of the coarse grid: each path returns the NaN status at the
    same step of one call and holds NaN at the same places of that step's top"""
    out = []
    for band2 in "012":
        monkeypatch.setenv("DNSG_BAND2", band2)
        s = dnsg.Solver(dnsg.make_params(xdv=40, ydv=9, zdv=12, gratio=2, zds=5, tau_c=0.53, ub=0.05, force_mode=force,
                                         g_const=2e-5, CFL=1.0, precision=prec, init_kind="laminar_noise", seed=5,
                                         u_max=0.05, noise=0.1))
        s.init_state()
        st = s.download()
        st["coarse"][20, 3, 6, 0] = np.nan
        s.upload(st["coarse"], st["lower"], st["upper"], st["lin"], st["uin"], st["force"])
        d = (dnsg.Diag * 60)()
        assert s.lib.dnsg_step(s.h, 60, d) == -3
        out.append((s.lib.dnsg_last_error(s.h).decode(), {k: np.isnan(v) for k, v in s.download().items() if k != "force"}))
        s.close()
    for msg, nan in out[1:]:
        assert msg == out[0][0]
        for k in KEYS:
            assert np.array_equal(nan[k], out[0][1][k]), k
