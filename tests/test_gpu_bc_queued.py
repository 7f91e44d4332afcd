"""ostc_zone_set_bc against boundary passes that are queued or captured: a
pass keeps the faces, wall flags and wall temperatures it was launched with,
and a queued one also its inflow states, whichever stream it waits on.  The
stream is one that does not wait for the null stream; copies hold it back
while the host sets the next program.

Equality is exact: the same kernels on the same state."""
import copy
import ctypes as C

import numpy as np
import pytest
import torch

from openstc_amd import _lib as L
from openstc_amd import cases
from openstc_amd.runtime import Simulation

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def make(kind):
    if kind == "plate":
        return cases.sst_plate(37, 21, 9, precision=L.FP32, perturb=True)
    return cases.mixing_layer(mx=21, my=18, mz=9, precision=L.FP64)


def changed(bc, inflow):
    """Another program: hot isothermal walls, the last face gone, the first
    symmetry face an outflow, and on request other inflow states."""
    b = copy.deepcopy(bc)
    for w in b.wall:
        w.isothermal, w.temperature = 1, 777.0
    b.n_face -= 1
    sym = [f for f in range(b.n_face) if b.face[f].kind == 3]
    b.face[sym[0]].kind = 6
    if inflow:
        for q in b.inflow:
            q.density, q.u, q.pressure = q.density * 1.25, q.u * 1.5, q.pressure * 1.75
    return b


def apply(sim, stream=None):
    L.check(sim.ctx.lib.ostc_apply_bc(sim.ctx.h, sim.zones[0].h, stream), "apply_bc")


def fields(sim):
    sim.sync()
    return [sim.zones[0].download(f) for f in ("BV", "SV", "CV")]


def start(kind):
    sim = Simulation(make(kind))
    sim.initialize_computation()
    sim.step()
    sim.sync()
    return sim


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("kind", ["plate", "mixing"])
def test_queued_pass_keeps_its_program(kind):
    print(f"[gpu-bc] queued pass, {kind}", flush=True)
    ref, sim = start(kind), start(kind)
    first = ref.zones[0]._bc
    second = changed(first, inflow=True)
    mid = changed(first, inflow=True)
    mid.n_face = first.n_face
    for s in (ref, sim):  # so that applying `first` again changes the ghosts
        s.zones[0].set_bc(mid)
        apply(s)
        s.sync()
        s.zones[0].set_bc(first)
    apply(ref)
    want_first = fields(ref)
    ref.zones[0].set_bc(second)
    apply(ref)
    want_second = fields(ref)
    assert not same(want_first, want_second)

    lib, n = sim.ctx.lib, 512 * MIB
    src, dst = C.c_void_p(), C.c_void_p()
    L.check(lib.ostc_device_alloc(C.byref(src), n), "alloc")
    L.check(lib.ostc_device_alloc(C.byref(dst), n), "alloc")
    stream = torch.cuda.Stream()
    st = C.c_void_p(stream.cuda_stream)
    sim.sync()
    for _ in range(64):
        L.check(lib.ostc_stream_copy(dst, src, n, st), "copy")
    apply(sim, st)
    sim.zones[0].set_bc(second)
    assert same(fields(sim), want_first)
    apply(sim, st)
    assert same(fields(sim), want_second)
    lib.ostc_device_free(src)
    lib.ostc_device_free(dst)
    ref.close()
    sim.close()


@pytest.mark.parametrize("kind", ["plate", "mixing"])
def test_captured_pass_keeps_its_faces_and_walls(kind):
    print(f"[gpu-bc] captured pass, {kind}", flush=True)
    sim = start(kind)
    z = sim.zones[0]
    before = fields(sim)
    first, second = z._bc, changed(z._bc, inflow=False)
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        apply(sim, C.c_void_p(torch.cuda.current_stream().cuda_stream))

    def restored():
        for f, a in zip(("BV", "SV", "CV"), before):
            if a.size:
                z.upload(f, a)
        sim.sync()

    # from a state whose ghosts are neither program's, so that every pass counts
    before[0] *= 1.01
    restored()
    apply(sim)
    want = fields(sim)
    z.set_bc(second)
    restored()
    apply(sim)
    other = fields(sim)
    assert not same(want, other)
    for k in range(4):
        restored()
        graph.replay()
        torch.cuda.synchronize()
        assert same(fields(sim), want), k
        restored()
        apply(sim)  # eager work between the replays
        assert same(fields(sim), other), k
    z.set_bc(first)
    sim.close()
