"""Snapshots into pageable arrays against pinned ones, at sizes on either side of the switch
to two pinned pieces of 16 MiB (from two pieces on) and with last pieces of every kind:
grid 0's velocity takes 24 bytes and its density 8 bytes a node of x y z."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import dnsg

pytestmark = pytest.mark.gpu
PIECE = 1 << 24


# x, y, z; bytes of the last piece of (velocity, density); None: a plain copy
@pytest.mark.parametrize("x,y,z,last", [
    (256, 128, 42, (None, None)),           # 33.03 MB, just below two pieces
    (256, 128, 43, (262144, None)),         # 33.82 MB, just beyond
    (256, 128, 128, (0, 0)),                # six and two whole pieces
    (117, 383, 78, (112, None)),            # five pieces and 112 bytes
])
def test_pageable_and_pinned_agree(x, y, z, last):
    for c, n in zip((24, 8), last):
        b = c * x * y * z
        assert (n is None) == (b < 2 * PIECE) and (n is None or n == b % PIECE)
    s = dnsg.Solver(dnsg.make_params(xdv=x, ydv=y, zdv=z, gratio=1, zds=4, tau_c=0.53, ub=0.05, force_mode="const",
                                     g_const=2e-5, CFL=1.0, init_kind="laminar_noise", seed=3, u_max=0.05, noise=0.1))
    s.init_state()
    s.step(1)
    vel, den = s.velocity(0)
    pv = torch.empty(vel.shape, dtype=torch.float64, pin_memory=True)
    pd = torch.empty(den.shape, dtype=torch.float64, pin_memory=True)
    ptr = lambda t: ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_double))
    s._check(s.lib.dnsg_velocity_snapshot(s.h, 0, ptr(pv), ptr(pd)))
    s.close()
    assert np.array_equal(vel, pv.numpy()) and np.array_equal(den, pd.numpy())
    assert np.isfinite(vel).all() and (den > 0.5).all()
