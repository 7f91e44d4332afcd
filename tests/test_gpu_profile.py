"""Stage timing covers what a time step launches: the part of an iteration
outside every bracket stays the same when the implicit sweeps are added."""
import ctypes as C

import pytest
import torch

from openstc_amd import _lib as L
from openstc_amd import cases
from openstc_amd.runtime import Simulation

pytestmark = pytest.mark.gpu


def outside_brackets(sweeps):
    """Milliseconds of an iteration that no stage accounts for (least of 8)."""
    sim = Simulation(cases.mixing_layer(mx=192, my=128, mz=96, precision=L.FP32, dplur_steps=sweeps))
    sim.initialize_computation()
    lib, n = sim.ctx.lib, sim.ctx.lib.ostc_profile_stage_count()
    ms, count = (C.c_double * n)(), (C.c_longlong * n)()
    for _ in range(3):
        sim.step()
    sim.sync()
    L.check(lib.ostc_profile(sim.ctx.h, 1), "profile")
    left = []
    for _ in range(8):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        sim.step()
        b.record()
        b.synchronize()
        L.check(lib.ostc_profile_read(sim.ctx.h, ms, count, n, 1), "profile_read")
        left.append(a.elapsed_time(b) - sum(ms))
    L.check(lib.ostc_profile(sim.ctx.h, 0), "profile off")
    sim.close()
    return min(left)


def test_sweeps_are_inside_brackets():
    """The bound: one bracket more costs its two events, under 0.02 ms; the
    pass that prepares the sweeps takes 0.1 ms on these 2.4 M cells."""
    none, one = outside_brackets(0), outside_brackets(1)
    print(f"[gpu-prof] outside the brackets: {none:.4f} ms without sweeps, {one:.4f} ms with one", flush=True)
    assert one - none < 0.05
