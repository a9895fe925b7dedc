"""A non-finite interface level of a checkpoint reaches what the method says, and no more.

Flux control: a NaN in the level before the newest enters the bands' interface layer with
the fills of the first step and spreads from there, by the end of that step over layers
that encalc2 gives no weight (encalc2.c:37-105: the bands overlap the coarse grid in
gratio layers).  The force of the second step is therefore bit for bit that of the run
without the NaN: the same sums over the same values.  Each form of the sums is run: the
two-substep band kernel, the aligned, paired and flat collide-stream forms, gratio 2 to 4.

Interface fill: the older levels carry the weight 0 at the last substep, and 0 x NaN is NaN
(tinterpolate_hrmt.c:28-34 forms every product), so the fills of the two steps that still
read uploaded levels leave NaN at the coarse nodes that hold one; the oldest
of the three uploaded levels is read by none."""
import numpy as np
import pytest

from helpers import dnsg

pytestmark = pytest.mark.gpu

# coarse x, gratio, precision, DNSG_BAND2
FLUX = [(20, 2, "fp64", "1"), (20, 2, "fp16", "1"), (256, 2, "fp32", "1"), (256, 2, "fp64", "0"), (256, 2, "fp32", "0"),
        (20, 2, "fp64", "0"), (20, 2, "fp16", "0"), (15, 3, "fp64", "0"), (64, 4, "fp64", "0"), (21, 4, "fp32", "0")]


def solver(x, gr, prec, level=None, value=np.nan, **kw):
    """a handle restarted from its own start, one value of both older-level stacks replaced"""
    s = dnsg.Solver(dnsg.make_params(xdv=x, ydv=10, zdv=10, gratio=gr, zds=8, tau_c=0.53, ub=0.05, CFL=1.0, precision=prec,
                                     init_kind="laminar_noise", seed=4, u_max=0.05, noise=0.1, **kw))
    s.init_state()
    st = s.download()
    if level is not None:
        for k in ("lin", "uin"):
            st[k][level, 7, 4, 0] = value
    s.upload(st["coarse"], st["lower"], st["upper"], st["lin"], st["uin"], st["force"])
    return s


@pytest.mark.parametrize("x,gr,prec,band2", FLUX)
def test_layers_without_weight_stay_out_of_the_force(x, gr, prec, band2, monkeypatch):
    monkeypatch.setenv("DNSG_BAND2", band2)
    a, b = solver(x, gr, prec, 0), solver(x, gr, prec)
    da, db = a.step(2), b.step(2)
    st = a.download()
    a.close(), b.close()
    assert np.isnan(st["lower"]).any() and np.isnan(st["upper"]).any()
    for f in ("force", "momentum", "density", "flowrate"):
        assert np.isfinite(da[f]).all() and np.array_equal(da[f], db[f]), f


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("gr,prec,level,steps", [(1, "fp64", 1, 1), (1, "fp32", 0, 2), (2, "fp64", 1, 1), (2, "fp16", 0, 2),
                                                 (3, "fp64", 0, 1), (4, "fp64", 1, 1)])
def test_uploaded_levels_reach_the_last_fill(gr, prec, level, steps, value):
    s = solver(20, gr, prec, level, value, force_mode="const", g_const=1e-5)
    s.step(steps)
    st = s.download()
    s.close()
    x, y = 7 * gr, 4 * gr
    assert np.isnan(st["lower"][x, y, -1]).all() and np.isnan(st["upper"][x, y, 0]).all()


@pytest.mark.parametrize("gr", [1, 2])
def test_own_levels_do_not(gr):
    """a NaN in the oldest uploaded level is read by no fill: one step later it is the spare"""
    a, b = solver(20, gr, "fp64", 2, force_mode="const", g_const=1e-5), solver(20, gr, "fp64", force_mode="const", g_const=1e-5)
    a.step(3), b.step(3)
    sa, sb = a.download(), b.download()
    a.close(), b.close()
    for k in ("coarse", "lower", "upper", "lin", "uin"):
        assert np.array_equal(sa[k], sb[k]), k
