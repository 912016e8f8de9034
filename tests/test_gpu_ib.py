"""GPU parity of the immersed-boundary, geometry and structural operators
(vivsim_amd.ib / ib3d / dyn) against the oracle."""

import math

import numpy as np
import pytest
import torch

from oracle import dyn as OD
from oracle import ib as OI
from tests.gpu_util import assert_close, dev, to_np

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(4242)


@pytest.fixture(scope="module")
def V(gpu_lib):
    import vivsim_amd
    return vivsim_amd


@pytest.mark.parametrize("name", ["peskin_2pt", "peskin_3pt", "peskin_4pt", "cosine_4pt"])
def test_kernels(V, name):
    r = np.linspace(-2.6, 2.6, 1001).astype(np.float32)
    got = getattr(V.ib, "kernel_" + name)(dev(r))
    assert_close(got, OI.KERNELS[name](r.astype(np.float64)), 2e-6, name)


@pytest.mark.parametrize("kernel,radius", [("peskin_4pt", 2), ("peskin_3pt", 2), ("cosine_4pt", 2),
                                           ("peskin_2pt", 1), ("peskin_4pt", 3)])
def test_stencil2d(V, kernel, radius):
    mx = (10 + 30 * rng.random(300)).astype(np.float32)
    my = (5 + 40 * rng.random(300)).astype(np.float32)
    W, I = V.ib.get_ib_stencil(dev(mx), dev(my), 57, kernel=getattr(V.ib, "kernel_" + kernel), stencil_radius=radius)
    W0, I0 = OI.get_ib_stencil(mx, my, 57, OI.KERNELS[kernel], radius)      # float32 oracle: same rounding
    assert np.array_equal(to_np(I), I0)
    assert_close(W, OI.get_ib_stencil(mx.astype(np.float64), my.astype(np.float64), 57, OI.KERNELS[kernel], radius)[0],
                 3e-6, "weights")
    assert W0.dtype == np.float32


def test_stencil3d(V):
    mc = (6 + 10 * rng.random((200, 3))).astype(np.float32)
    W, I = V.ib3d.get_ib_stencil(dev(mc), (24, 20, 22))
    W0, I0 = OI.get_ib_stencil3d(mc, (24, 20, 22))
    assert np.array_equal(to_np(I), I0)
    assert_close(W, OI.get_ib_stencil3d(mc.astype(np.float64), (24, 20, 22))[0], 3e-6, "weights3d")
    with pytest.raises(ValueError):
        V.ib3d.get_ib_stencil(dev(mc), (24, 20))
    with pytest.raises(ValueError):
        V.ib3d.get_ib_stencil(dev(mc[:, :2]), (24, 20, 22))


def test_interp_spread_mdf(V):
    nx, ny = 48, 40
    th = 2 * np.pi * np.arange(96) / 96
    mx = (24 + 9 * np.cos(th)).astype(np.float32)
    my = (20 + 9 * np.sin(th)).astype(np.float32)
    W, I = OI.get_ib_stencil(mx, my, ny)
    u = (0.05 * rng.standard_normal((2, nx, ny))).astype(np.float32)
    W64 = W.astype(np.float64)
    got = V.ib.interpolate(dev(u), dev(W), torch.as_tensor(I).cuda())
    assert_close(got, OI.interpolate(u.astype(np.float64), W64, I), 3e-6, "interp")
    F = (1e-3 * rng.standard_normal((96, 2))).astype(np.float32)
    base = (0.01 * rng.standard_normal((2, nx, ny))).astype(np.float32)
    got = V.ib.spread(dev(F), dev(base), dev(W), torch.as_tensor(I).cuda())
    assert_close(got, OI.spread(F.astype(np.float64), base.astype(np.float64), W64, I), 3e-6, "spread")
    U = np.zeros((96, 2), dtype=np.float32)
    U[:, 1] = 0.01
    ds = OI.get_ds(np.stack([mx, my], 1).astype(np.float64))
    for n_iter in (0, 1, 3):
        g, h = V.ib.multi_direct_forcing(dev(u), dev(W), torch.as_tensor(I).cuda(), dev(U), dev(ds), n_iter)
        g0, h0 = OI.multi_direct_forcing(u.astype(np.float64), W64, I, U.astype(np.float64), ds, n_iter)
        if n_iter == 0:
            assert torch.all(g == 0) and torch.all(h == 0)
        else:
            assert_close(g, g0, 2e-5, "mdf g")
            assert_close(h, h0, 2e-5, "mdf h")
    g, h = V.ib.multi_direct_forcing(dev(u), dev(W), torch.as_tensor(I).cuda(), dev(U), 0.6, 2)
    g0, h0 = OI.multi_direct_forcing(u.astype(np.float64), W64, I, U.astype(np.float64), 0.6, 2)
    assert_close(h, h0, 2e-5, "mdf scalar ds")


def test_out_of_range_indices(V):
    grid = np.arange(24, dtype=np.float32).reshape(2, 3, 4)
    W = np.ones((2, 3), dtype=np.float32)
    I = np.array([[-1, 12, 5], [13, -20, 0]], dtype=np.int32)
    assert_close(V.ib.interpolate(dev(grid), dev(W), torch.as_tensor(I).cuda()),
                 OI.interpolate(grid.astype(np.float64), W.astype(np.float64), I), 0, "clamp/wrap")
    mv = np.ones((2, 2), dtype=np.float32)
    got = V.ib.spread(dev(mv), dev(np.zeros((2, 3, 4), np.float32)), dev(W), torch.as_tensor(I).cuda())
    ref = OI.spread(mv.astype(np.float64), np.zeros((2, 3, 4)), W.astype(np.float64), I)
    assert np.array_equal(to_np(got), ref)


def test_geometry(V):
    N, R = 128, 12.0
    th = 2 * np.pi * np.arange(N) / N
    p = np.stack([30 + R * np.cos(th), 40 + R * np.sin(th)], 1).astype(np.float32)
    assert_close(V.ib.get_area(dev(p)).reshape(1), [OI.get_area(p.astype(np.float64))], 1e-6, "area")
    assert_close(V.ib.get_ds(dev(p)), OI.get_ds(p.astype(np.float64)), 1e-6, "ds closed")
    assert_close(V.ib.get_ds(dev(p), closed=False), OI.get_ds(p.astype(np.float64), closed=False), 1e-6, "ds open")
    v = rng.random((30, 3)).astype(np.float32)
    f = rng.integers(0, 30, size=(40, 3)).astype(np.int32)
    v64 = v.astype(np.float64)
    assert_close(V.ib3d.get_triangle_areas(dev(v), f), OI.get_triangle_areas(v64, f), 1e-6, "tri")
    assert_close(V.ib3d.get_surface_area(dev(v), f).reshape(1), [OI.get_surface_area(v64, f)], 1e-6, "surf")
    assert_close(V.ib3d.get_volume(dev(v), f).reshape(1), [OI.get_volume(v64, f)], 1e-5, "vol")
    assert_close(V.ib3d.get_ds(dev(v), f), OI.get_ds3d(v64, f), 1e-6, "vertex ds")


def test_dyn(V):
    a, v, d, h = np.array([0.1, -0.2]), np.array([0.3, 0.05]), np.array([0.0, 0.5]), np.array([0.05, 0.01])
    got = V.dyn.newmark(a, v, d, h, 2.0, 0.7, 0.1)
    ref = OD.newmark(a, v, d, h, 2.0, 0.7, 0.1)
    for x, y in zip(got, ref):
        assert np.allclose(to_np(x), y, rtol=1e-14, atol=1e-15)
    M, K, C = np.diag([2.0, 3.0]) + 0.1, np.array([[0.5, 0.1], [0.1, 0.7]]), np.diag([0.1, 0.0])
    got = V.dyn.newmark(a, v, d, h, M, K, C, dt=0.5)
    ref = OD.newmark(a, v, d, h, M, K, C, dt=0.5)
    for x, y in zip(got, ref):
        assert np.allclose(to_np(x), y, rtol=1e-12, atol=1e-14)
    s = V.dyn.newmark(0.1, 0.2, 0.3, 0.4, 1.0, 2.0, 0.0)
    assert np.isclose(float(s[2]), OD.newmark(0.1, 0.2, 0.3, 0.4, 1.0, 2.0, 0.0)[2])
    th = 2 * np.pi * np.arange(64) / 64
    x0, y0 = (5 + np.cos(th)).astype(np.float32), (6 + np.sin(th)).astype(np.float32)
    dd = np.array([0.1, -0.2, 0.3])
    xs, ys = V.dyn.get_markers_coords_3dof(dev(x0), dev(y0), 5.0, 6.0, dd)
    xr, yr = OD.get_markers_coords_3dof(x0.astype(np.float64), y0.astype(np.float64), 5.0, 6.0, dd)
    assert np.allclose(to_np(xs), xr, atol=2e-6) and np.allclose(to_np(ys), yr, atol=2e-6)
    x2, y2 = V.dyn.get_markers_coords_2dof(dev(x0), dev(y0), dd[:2])
    assert np.allclose(to_np(x2), x0 + 0.1, atol=1e-6) and np.allclose(to_np(y2), y0 - 0.2, atol=1e-6)
    vm = V.dyn.get_markers_velocity_3dof(xs, ys, 5.0, 6.0, dd, np.array([0.01, 0.02, 0.5]))
    assert np.allclose(to_np(vm), OD.get_markers_velocity_3dof(xr, yr, 5.0, 6.0, dd, np.array([0.01, 0.02, 0.5])),
                       atol=2e-6)
    hm = (0.1 * rng.standard_normal((64, 2))).astype(np.float32)
    assert np.allclose(to_np(V.dyn.get_force_to_obj(dev(hm))), hm.astype(np.float64).sum(0), rtol=1e-12, atol=1e-12)
    tq = V.dyn.get_torque_to_obj(dev(x0), dev(y0), 5.0, 6.0, np.zeros(3), dev(hm))
    assert math.isclose(float(tq), OD.get_torque_to_obj(x0.astype(np.float64), y0.astype(np.float64), 5.0, 6.0,
                                                        np.zeros(3), hm.astype(np.float64)), rel_tol=1e-6)
