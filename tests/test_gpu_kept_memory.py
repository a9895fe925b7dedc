"""Device memory that the library keeps between the calls that write results out."""
import numpy as np
import pytest
import torch

from helpers import dnsg

pytestmark = pytest.mark.gpu
MB = 1 << 20


def channel(x, y, z, **kw):
    s = dnsg.Solver(dnsg.make_params(xdv=x, ydv=y, zdv=z, gratio=2, zds=8, tau_c=0.53, ub=0.05, force_mode="const",
                                     g_const=2e-5, CFL=1.0, init_kind="laminar_noise", seed=3, u_max=0.05, noise=0.1, **kw))
    s.init_state()
    s.step(1)
    return s


def free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_release():
    """another allocator finds the memory after release_memory(), with the handle alive,
    and the next call gives the same results"""
    s = channel(256, 128, 96)
    a = s.budget2d()[:3]  # 32 bytes a node: 256 x 128 x 96 coarse, 2 x 512 x 256 x 9 fine
    nodes = 256 * 128 * 96 + 2 * 512 * 256 * 9
    before = free()
    dnsg.release_memory()
    assert free() - before >= 32 * nodes
    for u, v in zip(a, s.budget2d()[:3]):
        assert np.array_equal(u, v)
    s.close()


def test_coarse_spectra_keep_no_wall_layers():
    """the coarse grid has no wall layer: its spectra leave the handle without the device
    copies of the bands' (2 x 512 x 256 x 19 doubles), which a band's spectra read"""
    wall = 2 * 512 * 256 * 19 * 8
    first = channel(256, 128, 12)  # what the first use of a plan's kernels keeps
    first.spectra(0), first.spectra(1)
    s = channel(256, 128, 12)
    dnsg.release_memory()
    before = free()
    s.spectra(0)
    dnsg.release_memory()
    assert before - free() < wall // 2
    s.spectra(1)
    dnsg.release_memory()
    assert before - free() >= wall
    s.close(), first.close()
