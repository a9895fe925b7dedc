"""Large host copies go through two pinned pieces of 16 MiB by several threads; smaller
ones, and ones into memory the device can write, are plain copies.  Both move the same
bytes: snapshots of one state into a pageable and into a pinned array are equal, at sizes
below two pieces, of several pieces with a remainder, and of one byte row more than
whole pieces; spectra with a kept plan are those of a fresh handle."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import dnsg

pytestmark = pytest.mark.gpu


# grid 0: x y (z+2) nodes of 24 bytes: 31.9 MB (plain), 41 MB, and 2^25 bytes and a bit over
@pytest.mark.parametrize("x,y,z", [(190, 100, 68), (211, 97, 82), (256, 156, 34)])
def test_pageable_and_pinned_agree(x, y, z):
    p = dnsg.make_params(xdv=x, ydv=y, zdv=z, gratio=1, zds=4, tau_c=0.53, ub=0.05, force_mode="const", g_const=2e-5,
                         CFL=1.0, init_kind="laminar_noise", seed=3, u_max=0.05, noise=0.1)
    s = dnsg.Solver(p)
    s.init_state()
    s.step(1)
    vel, den = s.velocity(0)
    pv = torch.empty(vel.shape, dtype=torch.float64, pin_memory=True)
    pd = torch.empty(den.shape, dtype=torch.float64, pin_memory=True)
    ptr = lambda t: ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_double))
    s._check(s.lib.dnsg_velocity_snapshot(s.h, 0, ptr(pv), ptr(pd)))
    assert np.array_equal(vel, pv.numpy()) and np.array_equal(den, pd.numpy())
    assert np.isfinite(vel).all() and (den > 0.5).all()
    s.close()


@pytest.mark.parametrize("prec", ["fp64", "fp16"])
def test_kept_plan(prec):
    kw = dict(xdv=36, ydv=20, zdv=12, gratio=2, zds=5, tau_c=0.53, ub=0.05, force_mode="const", g_const=2e-5, CFL=1.0,
              precision=prec, init_kind="laminar_noise", seed=3, u_max=0.05, noise=0.1)
    s, f = dnsg.Solver(dnsg.make_params(**kw)), dnsg.Solver(dnsg.make_params(**kw))
    s.init_state(), f.init_state()
    for g in (2, 0, 1, 0):  # plans of the state before
        s.spectra(g)
    s.step(4), f.step(4)
    for g in range(3):
        for a, b in zip(s.spectra(g), f.spectra(g)):
            assert np.array_equal(a, b)
    s.close(), f.close()


def test_kept_blocks_between_handles_and_threads():
    """two handles of unlike sizes write their results from two threads at once, ten times,
    through one set of kept blocks: each result is the one that the handle gives alone"""
    from threading import Thread

    def solver(x, prec):
        s = dnsg.Solver(dnsg.make_params(xdv=x, ydv=24, zdv=14, gratio=2, zds=5, tau_c=0.53, ub=0.05, force_mode="const",
                                         g_const=2e-5, CFL=1.0, precision=prec, init_kind="laminar_noise", seed=x,
                                         u_max=0.05, noise=0.1))
        s.init_state()
        s.step(2)
        return s

    def results(s):
        out = [a for g in range(3) for a in (*s.spectra(g), *s.velocity(g))]
        return out + list(s.budget2d()[:3]) + list(s.download().values())

    hs = [solver(40, "fp64"), solver(56, "fp32")]
    alone = [results(s) for s in hs]
    bad = []

    def work(i):
        for _ in range(10):
            bad.extend(not np.array_equal(a, b) for a, b in zip(results(hs[i]), alone[i]))

    th = [Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in th], [t.join() for t in th]
    assert len(bad) == 20 * len(alone[0]) and not any(bad)
    [s.close() for s in hs]
