"""Lattice layers of 2 GiB and more.  The two-substep band kernel's form for them at small
sizes (DNSG_BAND2=3) against one launch per substep, as for its other tiles: bit for bit
under a constant force, within the tier's rounding under the flux controller.  And the real
ones, bands of 4096 x 3456 nodes (FP16 8192 x 6912): each path the same statistics, bit for
bit (they are sums of the state in one fixed order); rows of no whole chunks by a start without noise, whose
layers must stay uniform and equal those of a small channel."""
import numpy as np
import pytest

from helpers import dnsg, relmax

pytestmark = pytest.mark.gpu
KEYS = ("coarse", "lower", "upper", "lin", "uin")


def run(monkeypatch, band2, n, prec, x, y, zds, pattern, force):
    monkeypatch.setenv("DNSG_BAND2", band2)
    s = dnsg.Solver(dnsg.make_params(xdv=x, ydv=y, zdv=9, gratio=2, zds=zds, tau_c=0.53, ub=0.05, force_mode=force,
                                     g_const=2e-5, CFL=1.0, precision=prec, pattern=pattern, gxplussize=1, wxplussize=1,
                                     gyplussize=1, wyplussize=1, init_kind="laminar_noise", seed=5, u_max=0.05, noise=0.1))
    s.init_state()
    rec = s.step(n)
    st = s.download()
    s.close()
    return st, rec


@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16"])
@pytest.mark.parametrize("x,y,zds,pattern", [(31, 5, 4, "none"), (63, 11, 4, "rslip"), (61, 4, 7, "sslip"),
                                             (125, 21, 4, "pslip")])
def test_constant_force(x, y, zds, pattern, prec, monkeypatch):
    (a, ra), (b, rb) = (run(monkeypatch, v, 5, prec, x, y, zds, pattern, "const") for v in "30")
    for k in KEYS:
        assert np.array_equal(a[k], b[k]), k
    for f in ("momentum", "density", "str_up", "str_down"):
        assert np.allclose(ra[f], rb[f], rtol=1e-10, atol=0), f


@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16"])
def test_flux_control(prec, monkeypatch):
    (a, ra), (b, rb) = (run(monkeypatch, v, 20, prec, 97, 11, 5, "pslip", "flux") for v in "30")
    tol = {"fp64": 1e-12, "fp32": 1e-5, "fp16": 1e-2}[prec]
    for k in ("coarse", "lower", "upper"):
        assert relmax(a[k], b[k]) <= tol, k
    assert np.max(np.abs(ra["force"] - rb["force"])) <= tol * 0.05


def large(x, y, gr, zds, noise, force="const", **kw):
    s = dnsg.Solver(dnsg.make_params(xdv=x, ydv=y, zdv=7, gratio=gr, zds=zds, tau_c=0.53, ub=0.05, force_mode=force,
                                     g_const=2e-5, CFL=1.0, init_kind="laminar_noise", seed=5, u_max=0.05, noise=noise, **kw))
    s.init_state()
    rec = s.step(2)
    out = s.statistics(), s.band_launch_substeps(), rec
    s.close()
    return out


def test_bands_of_2_gib(monkeypatch):
    """bands of 4096 x 3456 (2.15 GB a layer): the pass, and two launches of the aligned form"""
    got = []
    for band2 in ("", "0"):
        monkeypatch.setenv("DNSG_BAND2", band2)
        st, sub, rec = large(2048, 1728, 2, 4, 0.1)
        assert sub == (1 if band2 else 2)
        got.append((st, rec))
        print("bands of 2 GiB: done", repr(band2), flush=True)
    (a, ra), (b, rb) = got
    assert np.isfinite(a).all() and np.array_equal(a, b)
    for f in ("momentum", "density", "str_up", "str_down"):
        assert np.allclose(ra[f], rb[f], rtol=1e-9, atol=0), f


@pytest.mark.parametrize("force", ["const", "flux"])
def test_pairs_in_fp16_bands_of_2_gib(force, monkeypatch):
    """FP16 bands of 8192 x 6912 (2.15 GB a layer): two nodes a thread, and one"""
    got = []
    for pair in "10":
        monkeypatch.setenv("DNSG_CS_PAIRED", pair)
        st, sub, rec = large(4096, 3456, 2, 4, 0.1, precision="fp16", force=force)
        assert sub == 1
        got.append((st, rec))
        print("FP16 bands of 2 GiB: done", force, pair, flush=True)
    (a, ra), (b, rb) = got
    assert np.isfinite(a).all()
    if force == "const":
        assert np.array_equal(a, b)
    else:
        assert relmax(a, b) <= 1e-2 and np.max(np.abs(ra["force"] - rb["force"])) <= 1e-2 * 0.05


def test_rows_of_no_whole_chunks():
    """4097 x 3456 (2.15 GB a layer) at gratio 1, the coarse grid and the bands"""
    a, _, _ = large(4097, 3456, 1, 4, 0.0)
    b, _, _ = large(37, 24, 1, 4, 0.0)
    assert np.max(np.abs(a[[0, 1, 2, 7]] - b[[0, 1, 2, 7]])) <= 1e-12
    assert np.max(np.abs(a[[3, 4, 5]])) <= 1e-9
