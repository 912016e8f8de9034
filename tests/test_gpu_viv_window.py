"""GPU test of the pipelined VIV step with a body that carries its window across
tile edges: against the separate IB and bulk launches of the same steps."""

import numpy as np
import pytest
import torch

from tests.gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,storage,tol", [(2048, 2048, "f32", 1e-5), (2048, 1990, "f32", 1e-5), (1500, 1500, "f16s", 1e-3),
                                               (4096, 4096, "f16s", 1e-3)])
@pytest.mark.parametrize("d0", [0.96, 0.9, 0.8])
def test_moving_window_crosses_a_tile_edge(gpu_lib, nx, ny, storage, tol, d0):
    """The IB kernel of a step ends long before the pass beside it, and the body's
    slot it writes is the one that held the state before that pass: the pass must
    take its tile order from something that stays as it is until it ends.  The window's origin goes from 1021
    to 1022, where the first row of its tiles (of 4 rows) changes, in step 1, 2
    or 4 of 7.  A tile left out would keep the populations of two steps earlier:
    with velocities that differ by 0.02 from cell to cell some 1e-2 of the
    largest population.  (f32: rounding of different kernels over 7 steps, some
    1e-7 each; f16s: its codes, 1e-4 of a deviation, may round differently.)"""
    from vivsim_amd import lbm, sim
    pc = sim.VIVCase(nx=nx, ny=ny, cx=1051.0, cy=ny / 2, dof=(True, True), mass_ratio=50.0, perturb=0.4)
    assert pc.ib_x0 == 1021
    say(f"moving window {nx}x{ny} {storage} from {d0}")
    u = torch.as_tensor(pc.initial_u(), dtype=torch.float32, device="cuda")
    f0 = lbm.get_equilibrium(torch.ones((nx, ny), device="cuda"), u)
    out = []
    for fused in (True, False):
        s = sim.VIV2D(pc, storage=storage, fused=fused)
        assert s.ib.fused == (2 if fused else 0)
        s.set_body(v=(0.06, 0.0), d=(d0, 0.0))
        f, hd, hh = s.run(f0, 7)
        s.check()
        out.append((f, hd, int(s.win_origin[0])))
    (a, da, xa), (b, db, xb) = out
    assert xa == xb == 1022
    err = float((a - b).abs().max() / b.abs().max())
    say(f"max rel diff {err:.2e}")
    assert err < tol
    assert np.allclose(da.cpu(), db.cpu(), rtol=0, atol=1e-6)


@pytest.mark.parametrize("storage,tol", [("f32", 1e-5), ("f16s", 1e-3)])
def test_body_set_between_short_runs(gpu_lib, storage, tol):
    """Runs of 1, 2, 1 and 4 steps, the body moved by some cells before each: a run's
    first pass takes the window of the body it finds.  (Tolerances as above.)"""
    from vivsim_amd import lbm, sim
    nx, ny = 620, 600
    pc = sim.VIVCase(nx=nx, ny=ny, cx=300.0, cy=ny / 2, dof=(True, True), mass_ratio=50.0, perturb=0.4)
    say(f"body set between runs {storage}")
    u = torch.as_tensor(pc.initial_u(), dtype=torch.float32, device="cuda")
    f0 = lbm.get_equilibrium(torch.ones((nx, ny), device="cuda"), u)
    out = []
    for fused in (True, False):
        s = sim.VIV2D(pc, storage=storage, fused=fused)
        f, seen = f0, []
        for n, d in ((1, (0.3, 0.0)), (2, (5.97, -2.4)), (1, (-7.1, 3.0)), (4, (40.95, 11.2))):
            s.set_body(v=(0.02, 0.01), d=d)
            f, hd, hh = s.run(f, n)
            s.check()
            seen += [int(s.win_origin[0]), int(s.win_origin[1])]
        out.append((f, hd, seen))
    (a, da, xa), (b, db, xb) = out
    assert xa == xb
    err = float((a - b).abs().max() / b.abs().max())
    say(f"max rel diff {err:.2e}")
    assert err < tol
    assert np.allclose(da.cpu(), db.cpu(), rtol=0, atol=1e-6)
