"""GPU test of vsx_timer_start / vsx_timer_stop: one time per full step of a run,
whether a launch takes one step or several."""

import ctypes

import pytest
import torch

from tests.gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(30, 50), (256, 240), (1100, 1050), (24, 20, 28)])
@pytest.mark.parametrize("n", [1, 2, 6, 7, 20])
def test_one_time_per_full_step(gpu_lib, shape, n):
    """A run of n steps has n - 1 full steps (the others open with the collision and
    close with the streaming).  Their times are positive and add up to less than
    the whole run, host included; at most max_pairs of them come back."""
    from vivsim_amd import lbm, lbm3d, sim
    say(f"timer: {shape} {n} steps")
    m = sim.LBM(shape, 1.5)
    f = (lbm if len(shape) == 2 else lbm3d).get_equilibrium(torch.ones(shape, device="cuda"),
                                                            torch.zeros((len(shape),) + shape, device="cuda"))
    m.run(f, n)
    ms, got = (ctypes.c_float * 64)(), ctypes.c_int32(-1)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    for cap in (64, 4):
        assert gpu_lib.vsx_timer_start(cap) == 0
        e0.record()
        m.run(f, n)
        e1.record()
        assert gpu_lib.vsx_timer_stop(ms, cap, ctypes.byref(got)) == 0
        e1.synchronize()
        assert got.value == min(n - 1, cap)
        t = list(ms[:got.value])
        assert all(x > 0 for x in t)
        assert sum(t) < e0.elapsed_time(e1)
