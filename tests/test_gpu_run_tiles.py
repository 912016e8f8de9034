"""GPU tests of the multi-operation 2D runs: every tile shape and kind of store
against the single passes, bit for bit, and the grids that take these kernels
against the float64 oracle, with every collision, forcing and wall list."""

import numpy as np
import pytest
import torch

from oracle import lbm2d as O
from tests.gpu_util import assert_close, dev, say
from tests.test_gpu_step2d import WALLSETS, run_oracle

pytestmark = pytest.mark.gpu
COLLISIONS = ["bgk", "mrt", "kbc", "reg"]


@pytest.fixture(scope="module")
def sim(gpu_lib):
    from vivsim_amd import sim
    return sim


def rand_state(nx, ny, u0=0.04):
    rng = np.random.default_rng(1000 * nx + ny)
    rho = 1 + 0.02 * rng.standard_normal((nx, ny))
    u = u0 * rng.standard_normal((2, nx, ny))
    return (O.get_equilibrium(rho, u) + 1e-3 * rng.standard_normal((9, nx, ny))).astype(np.float32)


def forces(kind, shape, rng):
    """(LBM arguments, the same force for the oracle)"""
    if kind == "none":
        return {}, None
    if kind == "uniform":
        g = np.zeros((2,) + shape)
        g[0], g[1] = np.float32(2e-5), np.float32(-1e-5)
        return dict(forcing="guo", g_uniform=(2e-5, -1e-5)), g
    g = (2e-4 * rng.standard_normal((2,) + shape)).astype(np.float32)
    return dict(forcing=kind, g=dev(g)), g.astype(np.float64)


def single_passes(m, f, n):
    """collide, n - 1 full steps, stream: one launch each"""
    w0, w1 = (torch.empty_like(x) for x in m.work())
    m.step(f, w0, "collide", src_f32=True)
    for _ in range(n - 1):
        m.step(w0, w1, "full")
        w0, w1 = w1, w0
    out = torch.empty_like(f)
    m.step(w0, out, "stream", dst_f32=True)
    return out


@pytest.mark.parametrize("force", ["none", "uniform", "guo", "edm"])
@pytest.mark.parametrize("storage", ["f32", "f16s", "bf16s", "e3m12s"])
@pytest.mark.parametrize("shape,n", [((40, 41), 9), ((256, 256), 6), ((257, 256), 7), ((362, 361), 13), ((511, 500), 6),
                                     ((513, 500), 7), ((1300, 1027), 8)])
def test_tiles_equal_single_passes(sim, shape, n, storage, force):
    """Tiles of 16 x 16 (up to 256 of them: 256 x 256), 16 x 32 (up to 512: 511 x 500), 20 x 64 and, 16-bit
    storage, 40 x 64 (1300 x 1027); rows of whole 128-byte lines (256) and others."""
    rng = np.random.default_rng(n)
    kw, _ = forces(force, shape, rng)
    f0 = dev(rand_state(*shape))
    for k, (walls, coll) in enumerate([("mixed", "bgk"), ("channel", "mrt"), ("cavity_nee", "kbc"), ("none", "reg"),
                                       ("channel", "kbc"), ("mixed", "reg")]):
        say(f"tiles {shape} {n} steps {storage} {force} {coll} {walls}")
        m = sim.LBM(shape, 1.6, collision=coll, walls=WALLSETS[walls], storage=storage, **kw)
        assert torch.equal(m.run(f0, n), single_passes(m, f0, n)), (coll, walls)


@pytest.mark.parametrize("nx,ny,storage", [(2760, 2740, "f32"), (3880, 3872, "f16s")])
def test_streamed_tiles_equal_single_passes(sim, nx, ny, storage):
    """Work buffers above 256 MiB (the last-level cache): 7 steps in two launches, the first of which writes
    the field with non-temporal stores, against single passes, which do so too in FP32."""
    f0 = dev(rand_state(nx, ny))
    say(f"streamed tiles {nx}x{ny} {storage}")
    m = sim.LBM((nx, ny), 1.7, collision="mrt", walls=WALLSETS["mixed"], storage=storage)
    assert torch.equal(m.run(f0, 7), single_passes(m, f0, 7))


def test_streamed_single_pass(sim):
    """Single passes of a field above 256 MiB (non-temporal stores of the full step) against the oracle."""
    nx, ny, n, om = 2760, 2740, 2, 1.7
    f0 = rand_state(nx, ny)
    say("streamed single passes 2760x2740")
    m = sim.LBM((nx, ny), om, collision="kbc", walls=WALLSETS["mixed"])
    got = single_passes(m, dev(f0), n)
    assert_close(got, run_oracle(f0, n, om, WALLSETS["mixed"], "kbc", None, None), 2e-5, "streamed single passes")


@pytest.mark.parametrize("force", ["none", "uniform", "guo", "edm"])
@pytest.mark.parametrize("collision", COLLISIONS)
@pytest.mark.parametrize("walls", list(WALLSETS))
def test_runs_match_oracle(sim, walls, collision, force):
    """The wall lists, collisions and forcings of the small-grid tests on grids whose sides the multi-operation
    kernels take (three launches of 12 steps' operations; tolerance of those tests)."""
    nx, ny, n, om = 61, 53, 12, 1.7
    rng = np.random.default_rng(len(walls) + len(force))
    kw, g = forces(force, (nx, ny), rng)
    f0 = rand_state(nx, ny)
    say(f"run {nx}x{ny} {collision} {walls} {force}")
    got = sim.LBM((nx, ny), om, collision=collision, walls=WALLSETS[walls], **kw).run(dev(f0), n)
    ref = run_oracle(f0, n, om, WALLSETS[walls], collision, kw.get("forcing"), g)
    assert_close(got, ref, 2e-5, f"{collision}/{walls}/{force}")


@pytest.mark.parametrize("shape", [(61, 53), (270, 262)])
def test_wall_arrays_match_oracle(sim, shape):
    """Per-node wall values (an inflow profile, a wall density, a moving lid) in tiles of 16 x 16 and 16 x 32."""
    nx, ny = shape
    rng = np.random.default_rng(nx)
    y = (np.arange(ny) + 0.5) / ny
    prof = (0.06 * y * (1 - y) * 4).astype(np.float32)
    rho = (1 + 0.005 * rng.random(ny)).astype(np.float32)
    lid = (0.03 * rng.random(nx)).astype(np.float32)
    low = (0.02 * rng.random(nx)).astype(np.float32)
    walls = [dict(kind="nebb", mode="velocity", loc="left", ux_wall=prof), dict(kind="nee", mode="pressure", loc="right", rho_wall=rho),
             dict(kind="bb", loc="bottom", ux_wall=low), dict(kind="nee", mode="velocity", loc="top", ux_wall=lid)]
    f0 = rand_state(nx, ny)
    say(f"wall arrays {shape}")
    ours = [{k: dev(v) if isinstance(v, np.ndarray) else v for k, v in w.items()} for w in walls]
    ref_walls = [{k: v.astype(np.float64) if isinstance(v, np.ndarray) else v for k, v in w.items()} for w in walls]
    for storage in ("f32", "f16s"):
        m = sim.LBM(shape, 1.7, collision="mrt", walls=ours, storage=storage)
        got = m.run(dev(f0), 9)
        assert torch.equal(got, single_passes(m, dev(f0), 9)), storage
        if storage == "f32":
            assert_close(got, run_oracle(f0, 9, 1.7, ref_walls, "mrt", None, None), 2e-5, "wall arrays")
