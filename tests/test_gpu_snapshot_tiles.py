"""Velocity snapshots, spectra and the budget where their kernels' tiles end (32 columns, 8
layers, 256-column workgroups of 8 rows): grids smaller than, exactly and just beyond a
tile in each direction, odd spanwise extents, the thinnest bands (whose one-sided stencils
reach into the next row).

* velocity and density from the downloaded distributions in vel_print's order: bitwise in
  FP64 (the same sums);
* spectra against numpy's transform of those planes: 1e-12 of the largest value;
* budget profiles against the oracle on the same snapshot: 1e-10 of each profile's scale."""
import numpy as np
import pytest

from helpers import budget_scales, dnsg, oracle_budget

pytestmark = pytest.mark.gpu

EX = [0, 1, -1, 0, 0, 0, 0, 1, -1, -1, 1, 1, 1, -1, -1, 0, 0, 0, 0]
EY = [0, 0, 0, 1, -1, 0, 0, 1, 1, -1, -1, 0, 0, 0, 0, 1, 1, -1, -1]
EZ = [0, 0, 0, 0, 0, 1, -1, 0, 0, 0, 0, 1, -1, -1, 1, 1, -1, -1, 1]


def vel_print(f):
    u = [np.zeros(f.shape[:3]) for _ in range(3)]
    rho = np.zeros(f.shape[:3])
    for q in range(19):
        for c, e in enumerate((EX, EY, EZ)):
            u[c] = u[c] + e[q] * f[..., q]
        rho = rho + f[..., q]
    return np.stack([c / rho for c in u], axis=-1), rho


@pytest.mark.parametrize("x,y,z,zds,gr", [(32, 8, 8, 4, 1), (33, 17, 10, 7, 1), (128, 4, 9, 8, 2), (129, 9, 11, 4, 2),
                                          (11, 6, 17, 9, 3)])
def test_snapshot_tiles(x, y, z, zds, gr):
    p = dnsg.make_params(xdv=x, ydv=y, zdv=z, gratio=gr, zds=zds, Rebs=40.0, ub=0.03, CFL=1.0, force_mode="const",
                         g_const=2e-5, init_kind="laminar_noise", seed=3, u_max=0.05, noise=0.2)
    s = dnsg.Solver(p)
    s.init_state()
    s.step(5)
    st = s.download()
    snaps = {}
    for g, name in enumerate(("coarse", "lower", "upper")):
        vel, rho = vel_print(st[name])
        v, d = s.velocity(g)
        assert np.array_equal(v, vel) and np.array_equal(d, rho), name
        snaps[g] = (v, d)
        N0, N1 = v.shape[:2]
        c = np.fft.rfft2(np.moveaxis(v, (2, 3), (1, 0)), axes=(2, 3)) / (N0 * N1)
        c[:, :, 0, 0] = 0.0
        e = np.where(np.arange(N1 // 2 + 1) == 0, 0.5, 1.0) * np.abs(c) ** 2
        ex, ey = s.spectra(g)
        rx, ry = np.moveaxis(e.sum(axis=3), 1, 2), np.moveaxis(e.sum(axis=2), 1, 2)
        assert np.max(np.abs(ex - rx)) <= 1e-12 * np.max(rx), name
        assert np.max(np.abs(ey - ry)) <= 1e-12 * np.max(ry), name
    got, ref = s.budget2d(planes=True), oracle_budget(p, snaps, planes=True)
    for kind, a, b in zip(("turb", "vort", "ke"), got, ref):
        scale = budget_scales(kind, b)[:, None]
        assert np.all(np.abs(a - b) <= 1e-10 * scale + 1e-300), kind
    for a, b in zip(got[3], ref[3]):
        assert np.max(np.abs(a - b)) <= 1e-13
    s.close()
