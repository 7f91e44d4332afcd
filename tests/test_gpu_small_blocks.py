"""Mixture sweeps that gather their neighbours and boundary faces launched
together, on blocks thinner than a tile, a wave or the ghost layers: the halo
of one face then reaches the interior points of the opposite one, and every
tile has a remainder.  Against the FP64 oracle.

Tolerance: 1e-9 of each field's largest value after 2 iterations in FP64 (the
bound of the other trajectory tests; one operation is 1e-16 and an iteration
amplifies by the sweeps' 1e2..1e4).  The velocities have one scale: w of the
mixing layer is a perturbation of u and its rounding is u's.  Trace species
(below 1e-6 of the largest) are left out: what two iterations make of them is
a difference of rates, rounded relative to the rates (131x18x3 shows 1.4e-9
also without a single sweep)."""
import numpy as np
import pytest

from harness import Pair, interior, scaled_err
from openstc_amd import _lib as L
from openstc_amd import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(5, 4, 3), (64, 4, 4), (65, 9, 5), (67, 3, 26), (131, 18, 3)])
@pytest.mark.parametrize("sweeps", [0, 1, 4])
def test_mixture_sweeps(shape, sweeps):
    print(f"[gpu-small] mixing layer {shape}, {sweeps} sweeps", flush=True)
    pr = Pair(cases.mixing_layer(mx=shape[0], my=shape[1], mz=shape[2], precision=L.FP64, dplur_steps=sweeps),
              precision=L.FP64)
    pr.init()
    for _ in range(2):
        pr.gpu.step()
        pr.orc.step()
    a, b = interior(pr.gpu.zones[0].download("BV")), interior(pr.orc.blocks[0].arr["bv"])
    e = max(scaled_err(a[[0, 4, 5]], b[[0, 4, 5]]), np.abs(a[1:4] - b[1:4]).max() / np.abs(b[1:4]).max())
    print(f"[gpu-small] flow err {e:.2e}", flush=True)
    a = interior(pr.gpu.zones[0].download("SV"))
    b = interior(pr.orc.blocks[0].arr["sv"][:len(a)])
    scale = np.abs(b).reshape(len(b), -1).max(1)
    big = scale > 1e-6 * scale.max()
    e = max(e, scaled_err(a[big], b[big]))
    print(f"[gpu-small] err {e:.2e}", flush=True)
    assert e < 1e-9
    pr.close()


@pytest.mark.parametrize("shape", [(3, 3, 3), (4, 70, 3), (9, 3, 5), (66, 5, 4)])
def test_faces(shape):
    print(f"[gpu-small] warped box {shape}", flush=True)
    pr = Pair(cases.warped_box(mx=shape[0], my=shape[1], mz=shape[2]))
    pr.init()
    for _ in range(2):
        pr.gpu.step()
        pr.orc.step()
    e = pr.err("BV", halo=2)
    print(f"[gpu-small] err {e:.2e}", flush=True)
    assert e < 1e-9
    pr.close()


@pytest.mark.parametrize("patches", [2, 5])
@pytest.mark.parametrize("mz", [5, 11])
def test_faces_in_patches(patches, mz):
    """Each face of a plate cut into patches, 10 and 30 faces a program: runs of
    disjoint ones longer than a launch takes, and between them faces that meet
    at an edge and keep their order (5 planes: the k faces meet as well)."""
    print(f"[gpu-small] plate 24x20x{mz}, {patches} patches a face", flush=True)
    case = cases.sst_plate(24, 20, mz, precision=L.FP64, cfl=2.0, perturb=True)
    whole, bc = case.blocks[0].bc, L.BC()
    bc.inflow, bc.wall = whole.inflow, whole.wall
    for f in range(whole.n_face):
        src = whole.face[f]
        along = 1 if src.face == 0 else 0
        lo, n = src.range_start[along], src.range_end[along] - src.range_start[along] + 1
        for q in range(patches):
            dst = bc.face[bc.n_face]
            bc.n_face += 1
            for k, _ in L.Face._fields_:
                setattr(dst, k, getattr(src, k))
            dst.range_start[along], dst.range_end[along] = lo + n * q // patches, lo + n * (q + 1) // patches - 1
    case.blocks[0].bc = bc
    pr = Pair(case, precision=L.FP64)
    pr.init()
    for step in range(3):
        e = max(pr.err("BV", halo=2), pr.err("SV", halo=2))
        print(f"[gpu-small] after {step} steps: err {e:.2e}", flush=True)
        assert e < 1e-9
        pr.gpu.step()
        pr.orc.step()
    pr.close()
