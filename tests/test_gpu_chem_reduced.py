"""The chemistry reduced by the conserved elements against the FP64 oracle,
which solves the whole species block: mechanisms of every shape its tables
take (few reactions, more than 20, species that only act as catalysts) and one
they do not take, which runs on the whole block.

Tolerances: the point step 1e-9 of the largest change of each state (FP64
exp/log differences, 1e-14 measured, times the block's condition number for
time steps up to 1e-5 s); FP32 zones after 3 iterations 2e-5, FP64 zones 1e-9
of each field's largest value, the bounds of the other trajectory tests."""
import ctypes as C

import numpy as np
import pytest

import oracle_ffi as O
from harness import Pair, interior, scaled_err
from openstc_amd import _lib as L
from openstc_amd import cases
from openstc_amd.runtime import Context, Simulation
from openstc_amd.surrogate import DeviceArray, Surrogate
from test_gpu_chem import Dev, states

pytestmark = pytest.mark.gpu
NS, NR = 20, 50  # strides of the species and reaction arrays
ARRAYS = ("A", "b", "Ea", "A2", "b2", "Ea2", "reac_type", "reac_order", "troe_alpha", "troe_t1", "troe_t2", "troe_t3")


def take(param, reactions):
    """param with these of its reactions, in this order (repeats allowed)."""
    rows = {k: list(getattr(param, k)) for k in ARRAYS + ("stoi_f", "stoi_b", "third_body_coeff")}
    for q, r in enumerate(reactions):
        for k in ARRAYS:
            getattr(param, k)[q] = rows[k][r]
        for k in ("stoi_f", "stoi_b", "third_body_coeff"):
            getattr(param, k)[q * NS:(q + 1) * NS] = rows[k][r * NS:(r + 1) * NS]
    param.n_reac = len(reactions)
    return param


def mechanism(name):
    mech, _ = cases.load_mechanism(True)
    if name == "one reaction":  # one kept row, three dependent ones: too many, the whole block
        return take(mech, [0])
    if name == "two kept rows":  # H+O2=O+OH and H+O+M=OH+M: H, O2, O, OH
        return take(mech, [0, 6])
    if name == "24 reactions":  # more than the rate table in LDS holds
        return take(mech, list(range(19)) + [1, 3, 5, 8, 10])
    if name == "inert catalyst":  # N2 takes part without changing: nine species react
        mech.stoi_f[2 * NS + 8] = mech.stoi_b[2 * NS + 8] = 1
        return mech
    return mech


NAMES = ["as shipped", "one reaction", "two kept rows", "24 reactions", "inert catalyst"]


def with_flow(mech):
    fs = cases.InflowState(1.0, 1.0, 0, 0, 1e5, 1000.0, 1.0, 0.0, [0.0] * 9)
    return cases.mixture_param(mech, False, True, 4, 1.0, 1, fs)


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("n", [1, 255, 1025])
def test_point_step(name, n):
    print(f"[gpu-red] point step, {name}, n={n}", flush=True)
    param = with_flow(mechanism(name))
    ctx = Context(param)
    t, p, y, dt = states(n, 5)
    y[0, 1] = y[0, 5] = 0.0  # absent species: zero columns
    dev = [Dev(a) for a in (t, p, y, dt, np.zeros((n, 9)))]
    L.check(ctx.lib.ostc_chem_plain_step(ctx.h, n, *(d.p for d in dev), None), "plain")
    got = dev[4].get()
    op, lib = O.copy_struct(O.OrcParam, param), O.load()
    want = np.zeros((n, 9))
    for c in range(n):
        yy, out = np.ascontiguousarray(np.pad(y[c], (0, 11))), np.zeros(20)
        lib.orc_plain_chem_step(C.byref(op), t[c], p[c], O.dp(yy), dt[c], O.dp(out))
        want[c] = out[:9]
    e = (np.abs(got - want).max(1) / (np.abs(want).max(1) + 1e-300)).max()
    print(f"[gpu-red] max rel err {e:.2e}", flush=True)
    assert e < 1e-9
    for d in dev:
        d.free()
    ctx.close()


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("precision,tol", [(L.FP64, 1e-9), (L.FP32, 2e-5)])
def test_time_step(name, precision, tol):
    """Three iterations of a mixing layer with each mechanism."""
    print(f"[gpu-red] mixing layer 21x18x9, {name}, precision {precision}", flush=True)
    case = cases.mixing_layer(mx=21, my=18, mz=9, precision=precision)
    mech = mechanism(name)
    for k in ARRAYS + ("stoi_f", "stoi_b", "third_body_coeff"):
        getattr(case.param, k)[:] = list(getattr(mech, k))
    case.param.n_reac = mech.n_reac
    pr = Pair(case, precision=precision)
    pr.init()
    for _ in range(3):
        pr.gpu.step()
        pr.orc.step()
    for f, o in (("BV", "bv"), ("SV", "sv"), ("CV", "cv")):
        a = interior(pr.gpu.zones[0].download(f))
        b = interior(pr.orc.blocks[0].arr[o][:a.shape[0]])
        if f == "BV":  # one velocity scale: w is a small perturbation
            a, b = np.stack([a[0], *a[1:4], a[4], a[5]]), np.stack([b[0], *b[1:4], b[4], b[5]])
            scale = np.abs(b[1:4]).max()
            e = max(scaled_err(a[[0, 4, 5]], b[[0, 4, 5]]), np.abs(a[1:4] - b[1:4]).max() / scale)
        else:
            scale = np.abs(b).reshape(len(b), -1).max(1)
            big = scale > 1e-6 * scale.max()
            e = scaled_err(a[big], b[big])
        print(f"[gpu-red] {f} err {e:.2e}", flush=True)
        assert e < tol, (f, e)
    pr.gpu.close()


@pytest.mark.parametrize("own,zone", [("as shipped", "inert catalyst"), ("inert catalyst", "as shipped")])
@pytest.mark.parametrize("precision", [L.FP64, L.FP32])
def test_fallback_takes_the_zones_mechanism(own, zone, precision):
    """A surrogate may step a zone of another context: the cells it rejects
    take the plain step of the zone's mechanism, with or without the tables."""
    print(f"[gpu-red] surrogate of '{own}' on a zone of '{zone}', precision {precision}", flush=True)
    sur = Surrogate.load(Context(with_flow(mechanism(own))), t_max=1.0)  # rejects every state
    case = cases.mixing_layer(mx=21, my=18, mz=9, precision=precision)
    mech = mechanism(zone)
    for k in ARRAYS + ("stoi_f", "stoi_b", "third_body_coeff"):
        getattr(case.param, k)[:] = list(getattr(mech, k))
    case.param.n_reac = mech.n_reac
    sim = Simulation(case)
    sim.initialize_computation()
    sim.step()
    n = 21 * 18 * 9
    dy, st = [DeviceArray(nbytes=n * 9 * 8) for _ in range(2)], (C.c_longlong * 4)()
    for mode in (0, 1):
        L.check(sim.ctx.lib.ostc_chem_zone_step(sim.ctx.h, sim.zones[0].h, sur.h if mode else None, mode, dy[mode].p,
                                                st if mode else None, None), "zone chemistry")
    plain, got = (d.get(np.float64, (n, 9)) for d in dy)
    assert list(st) == [n, n, 0, 0]
    assert np.abs(plain).max() > 0 and np.array_equal(got, plain)
    for d in dy:
        d.free()
    sur.close()
    sim.close()
