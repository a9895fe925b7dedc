"""The collide-stream form that rows of no whole chunks take in layers of 2 GiB and more (one
chunk of a row per workgroup, 64-bit addresses), which DNSG_CS_WIDE selects at any size: for the coarse grid, the bands or
both, so that it also shares a step with the other forms.

FP64 against the oracle: bit for bit under a constant force, 1e-12 of the largest value
under the flux controller (its sums are taken in another order).  Shifted tiers against the
forms they take by themselves: the same collisions on the same values, so bit for bit under
a constant force, and within the tier's rounding (1e-5, 1e-2 of the largest value) where the
force feeds back from the sums.  Rows shorter and longer than a chunk, of exactly one (the
aligned FP64 form otherwise) and of two (the paired form otherwise); each gratio; walls with
posts; the filtered injection; the batched launches of the queue."""
import numpy as np
import pytest

from helpers import Oracle, dnsg, relmax

pytestmark = pytest.mark.gpu

KEYS = ("coarse", "lower", "upper", "lin", "uin")
# coarse x, y, gratio
SHAPES = [(17, 6, 1), (256, 4, 1), (300, 2, 1), (8, 4, 2), (128, 3, 2), (512, 2, 2), (43, 5, 3), (33, 7, 4)]


def params(x, y, gr, prec, force, **kw):
    return dnsg.make_params(xdv=x, ydv=y, zdv=8, gratio=gr, zds=7, tau_c=0.53, ub=0.05, force_mode=force, g_const=2e-5,
                            CFL=1.0, precision=prec, pattern="pslip", gxplussize=gr * x - 1, wxplussize=1, gyplussize=1,
                            wyplussize=gr * y - 1, init_kind="laminar_noise", seed=9, u_max=0.05, noise=0.1, **kw)


def run(p, wide, monkeypatch, n=4):
    monkeypatch.setenv("DNSG_CS_WIDE", str(wide))
    s = dnsg.Solver(p)
    if wide & 2:
        assert s.band_launch_substeps() == 1
    s.init_state()
    rec = s.step(n)
    st = s.download()
    s.close()
    return st, rec


@pytest.mark.parametrize("force", ["const", "flux"])
@pytest.mark.parametrize("wide", [1, 2, 3])
@pytest.mark.parametrize("x,y,gr", SHAPES)
def test_fp64_against_oracle(x, y, gr, wide, force, monkeypatch):
    p = params(x, y, gr, "fp64", force)
    a, da = run(p, wide, monkeypatch)
    o = Oracle(p)
    o.init_seeded()
    do, b = o.run(4), o.state()
    for k in KEYS:
        if force == "const":
            assert np.array_equal(a[k], b[k]), k
        else:
            assert relmax(a[k], b[k]) <= 1e-12, k
    for f in ("momentum", "density", "str_up", "str_down"):
        assert np.allclose(da[f], do[f], rtol=1e-10, atol=1e-16), f


@pytest.mark.parametrize("force", ["const", "flux"])
@pytest.mark.parametrize("prec", ["fp32", "fp16"])
@pytest.mark.parametrize("x,y,gr", [(17, 6, 1), (128, 3, 2), (512, 2, 2), (33, 7, 4)])
def test_shifted_tiers(x, y, gr, prec, force, monkeypatch):
    p = params(x, y, gr, prec, force)
    ref, dr = run(p, 0, monkeypatch)
    tol = {"fp32": 1e-5, "fp16": 1e-2}[prec]
    for wide in (1, 2, 3):
        a, da = run(p, wide, monkeypatch)
        for k in KEYS:
            assert np.array_equal(a[k], ref[k]) if force == "const" else relmax(a[k], ref[k]) <= tol, (wide, k)
        for f in ("momentum", "density"):
            assert relmax(da[f], dr[f]) <= (1e-12 if force == "const" else tol), (wide, f)


def test_filtered_injection(monkeypatch):
    p = params(12, 6, 4, "fp64", "flux", fltr=1)
    a, _ = run(p, 3, monkeypatch)
    o = Oracle(p)
    o.init_seeded()
    o.run(4)
    b = o.state()
    for k in KEYS:
        assert relmax(a[k], b[k]) <= 1e-12, k


def test_queue(monkeypatch):
    """launches of several lattices, some wide and some not: the same bulk velocities"""
    got = []
    for wide in "013":
        monkeypatch.setenv("DNSG_CS_WIDE", wide)
        q = dnsg.Queue(max_steps=40, check_every=20, window=20, max_active=4)
        for i, gr in enumerate((1, 2, 2)):
            q.submit(dnsg.slip_request(32 + 16 * i, 16, 12, gr, "rslip", 8, 0.5, 50.0, precision="fp32", seed=i), i)
        done = []
        while len(done) < 3:
            done += q.advance(20)
        q.close()
        got.append({r["id"]: (r["steps"], r["ubulk"]) for r in done})
    for g in got[1:]:
        for i in range(3):
            assert g[i][0] == got[0][i][0] and abs(g[i][1] - got[0][i][1]) <= 1e-12 * abs(got[0][i][1])
