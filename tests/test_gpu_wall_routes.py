"""GPU parity of the pure wall functions on both sides of the field size at which
they change kernels (2 MB: one kernel that copies and applies the wall below it, a copy
and a wall kernel above), against the oracle: every location, the kinds that
read the neighbour line, the wall line only and the pre-streaming field, and per-node
values.  Tolerances are those of the single-operator tests (a few float32 ulps)."""

import numpy as np
import pytest

from oracle import lbm2d as O2
from oracle import lbm3d as O3
from tests.gpu_util import assert_close, dev, say

pytestmark = pytest.mark.gpu
LIMIT = 2 << 20
SHAPES = [(241, 239), (243, 241), (29, 31, 29), (31, 30, 33)]   # 2.07, 2.11, 1.98 and 2.33 million bytes


def test_shapes_lie_on_both_sides():
    size = [4 * (9 if len(s) == 2 else 19) * int(np.prod(s)) for s in SHAPES]
    assert size[0] <= LIMIT < size[1] and size[2] <= LIMIT < size[3]


def state(shape):
    rng = np.random.default_rng(sum(shape))
    O, q = (O2, 9) if len(shape) == 2 else (O3, 19)
    rho = 1 + 0.05 * rng.standard_normal(shape)
    u = 0.05 * rng.standard_normal((len(shape),) + shape)
    pre = (O.get_equilibrium(rho, u) + 2e-3 * rng.standard_normal((q,) + shape)).astype(np.float32)
    return rng, O, pre, O.streaming(pre)


def locations(shape):
    return ["left", "right", "bottom", "top"] + (["back", "front"] if len(shape) == 3 else [])


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_walls_on_both_sides(gpu_lib, shape):
    from vivsim_amd import lbm, lbm3d
    L = lbm if len(shape) == 2 else lbm3d
    rng, O, pre, fs = state(shape)
    uz = dict(uz_wall=0.01) if len(shape) == 3 else {}
    f64 = fs.astype(np.float64)
    for axis, loc in enumerate(locations(shape)):
        say(f"walls {shape} {loc}")
        for name, kw in [("boundary_nee", dict(rho_wall=1.01, ux_wall=0.03, uy_wall=-0.02, **uz)),
                         ("boundary_pressure_nee", dict(rho_wall=0.99)),
                         ("boundary_velocity_nebb", dict(ux_wall=0.05, uy_wall=-0.01, **uz)),
                         ("boundary_equilibrium", dict(rho_wall=1.0, ux_wall=0.05))]:
            got = getattr(L, name)(dev(fs), loc, **kw)
            assert_close(got, getattr(O, name)(f64, loc, **kw), 5e-6, f"{name} {loc}")
        for name in ("boundary_bounce_back", "boundary_specular_reflection"):
            got = getattr(L, name)(dev(pre), dev(fs), loc, ux_wall=0.02, uy_wall=-0.01)
            ref = getattr(O, name)(pre.astype(np.float64), f64, loc, ux_wall=0.02, uy_wall=-0.01)
            assert_close(got, ref, 3e-6, f"{name} {loc}")
        nodes = tuple(np.delete(shape, axis // 2))
        ux = (0.05 * rng.random(nodes)).astype(np.float32)
        rw = (1 + 0.01 * rng.random(nodes)).astype(np.float32)
        got = L.boundary_nee(dev(fs), loc, rho_wall=dev(rw), ux_wall=dev(ux), uy_wall=0.01)
        ref = O.boundary_nee(f64, loc, rho_wall=rw.astype(np.float64), ux_wall=ux.astype(np.float64), uy_wall=0.01)
        assert_close(got, ref, 5e-6, f"nee arrays {loc}")
