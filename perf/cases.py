"""Workloads that stand for what users of this framework run, with a plain
64-bit statement of what each one returns.

Two groups:

* whole steady iterations of the time loop (``Simulation.step``: sources,
  fluxes, time step, implicit treatment, update, boundary conditions, block
  exchange, properties) on the four model families: the Euler box, the SST
  plate, the finite-rate mixing layer and the multi-block jet with SST and
  finite-rate chemistry;
* the chemistry calls on batches of states: the plain point-implicit step, the
  learned surrogate that stands in for it, and the surrogate's gradients.

``exact`` restates them in float64 torch from the formulas alone (second-order
finite volumes on curvilinear blocks; nothing of the package's kernels).
"""
from __future__ import annotations

import ctypes as C
import math
import os

import numpy as np
import torch

from openstc_amd import _lib as L
from openstc_amd import cases as workloads
from openstc_amd import surrogate as sur
from openstc_amd.runtime import Context, Simulation

NO_RESIDUAL = 1 << 30  # output_screen: the residual is printed every this many steps
WEIGHTS = {"gelu": sur.DEFAULT_WEIGHTS, "hswish": sur.HSWISH_WEIGHTS}


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # the smallest call: one small FP64 block, explicit Euler; every kernel
        # is short, so launches and latency count
        dict(name="box_fp64", kind="box", mx=64, my=64, mz=8, blocks=1, precision=8),
        # the Euler path at an ordinary, ragged size, cut into two blocks
        dict(name="box_two_blocks_fp64", kind="box", mx=147, my=95, mz=41, blocks=2, precision=8),
        # turbulent wall flow, the benchmark's plate (FP32 bulk, DPLUR)
        dict(name="plate_fp32", kind="plate", mx=256, my=128, mz=64, steps=4, cfl=5.0, precision=4),
        # the same path in double precision on a ragged mesh
        dict(name="plate_fp64_ragged", kind="plate", mx=119, my=67, mz=31, steps=4, cfl=2.0, precision=8),
        # laminar finite-rate combustion, the benchmark's mixing layer
        dict(name="mixing_fp32", kind="mixing", mx=192, my=96, mz=96, steps=4, reacting=True, precision=4),
        # a coarse-mesh run of it, as one does to start or to test a case
        dict(name="mixing_coarse_fp32", kind="mixing", mx=57, my=41, mz=23, steps=4, reacting=True, precision=4),
        # mixing without reactions (species transport only)
        dict(name="mixing_inert_fp32", kind="mixing", mx=131, my=75, mz=53, steps=4, reacting=False, precision=4),
        # the full model on blocks: SST, finite-rate chemistry, block exchange;
        # the headline workload's four blocks at about 3/8 of its cells
        dict(name="jet_four_blocks_fp32", kind="jet", mx=192, my=128, mz=96, blocks=4, steps=4, precision=4),
        # the same model on small ragged blocks
        dict(name="jet_two_blocks_fp32", kind="jet", mx=75, my=52, mz=37, blocks=2, steps=4, precision=4),
        # point chemistry on a batch of states (labels for training, studies)
        dict(name="chemistry_batch", kind="chemistry", n=1000000),
        # surrogate inference with its checks and fallback, a large batch
        dict(name="surrogate_batch", kind="surrogate", n=1500000, weights="gelu"),
        # one training batch of the surrogate: loss gradients of all weights
        dict(name="surrogate_gradients", kind="gradients", n=4096, weights="gelu"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["box", "plate", "plate", "mixing", "mixing", "jet", "jet", "chemistry", "surrogate",
                       "gradients"])
    precision = rng.choice([4, 8])
    if kind == "box":
        return dict(kind=kind, mx=_log_int(rng, 24, 192), my=_log_int(rng, 16, 160), mz=_log_int(rng, 8, 64),
                    blocks=rng.choice([1, 2]), precision=precision)
    if kind == "plate":
        return dict(kind=kind, mx=_log_int(rng, 32, 288), my=_log_int(rng, 32, 144), mz=_log_int(rng, 8, 72),
                    steps=rng.choice([2, 4, 6]), cfl=rng.choice([2.0, 5.0]), precision=precision)
    if kind == "mixing":
        return dict(kind=kind, mx=_log_int(rng, 28, 200), my=_log_int(rng, 20, 112), mz=_log_int(rng, 8, 104),
                    steps=rng.choice([2, 4, 6]), reacting=rng.random() < 0.75, precision=precision)
    if kind == "jet":
        return dict(kind=kind, mx=_log_int(rng, 32, 160), my=_log_int(rng, 20, 128), mz=_log_int(rng, 16, 80),
                    blocks=rng.choice([2, 3, 4]), steps=rng.choice([2, 4]), precision=4)
    if kind == "gradients":
        return dict(kind=kind, n=16 * _log_int(rng, 16, 256), weights=rng.choice(["gelu", "hswish"]))
    if kind == "surrogate":
        return dict(kind=kind, n=_log_int(rng, 2000, 1500000), weights=rng.choice(["gelu", "hswish"]))
    return dict(kind=kind, n=_log_int(rng, 1000, 1000000))


def _flow_case(case, seed):
    """The workload's mesh, constants and perturbed initial field."""
    kind, prec = case["kind"], case["precision"]
    if kind == "box":
        if case["blocks"] == 1:
            return workloads.warped_box(case["mx"], case["my"], case["mz"], precision=prec, seed=seed)
        return workloads.warped_box_split(case["mx"], case["my"], case["mz"], precision=prec, seed=seed)
    if kind == "plate":
        return workloads.sst_plate(case["mx"], case["my"], case["mz"], precision=prec, dplur_steps=case["steps"],
                                   cfl=case["cfl"], seed=seed, perturb=True)
    if kind == "mixing":
        c = workloads.mixing_layer(case["mx"], case["my"], case["mz"], precision=prec, dplur_steps=case["steps"],
                                   seed=seed)
        if not case["reacting"]:
            c.param.mix_model = L.MIXTURE
        return c
    return workloads.jet_crossflow(case["mx"], case["my"], case["mz"], nblocks=case["blocks"], precision=prec,
                                   dplur_steps=case["steps"], seed=seed)


# ------------------------------------------------------------------ the calls

class _DeviceView:
    """A zone field as a torch tensor over the zone's own memory."""

    def __init__(self, zone, field):
        ptr, size, planes = C.c_void_p(), C.c_int(), zone.planes(field)
        L.check(zone.lib.ostc_zone_field_ptr(zone.h, L.F[field], C.byref(ptr), C.byref(size)), field)
        self.zone = zone
        self.__cuda_array_interface__ = dict(shape=(planes,) + zone.shape, typestr=f"<f{size.value}",
                                             data=(ptr.value, False), version=2)


def _interior(zone, field):
    g = zone.ngg
    return torch.as_tensor(_DeviceView(zone, field), device="cuda")[:, g:-g, g:-g, g:-g]


def _fields(param, bv, sv, cv, mul, lam, mut):
    """What an iteration leaves: the state, and the properties it carries on."""
    ns = param.n_spec
    out = dict(density=bv[0], velocity=bv[1:4], pressure=bv[4], temperature=bv[5], energy=cv[4], momentum=cv[1:4],
               viscosity=mul, conductivity=lam)
    if ns:
        out["species"] = sv[:ns]
    if param.turb_method == L.RANS:
        out["tke"], out["omega"], out["eddy_viscosity"] = sv[ns], sv[ns + 1], mut
    return out


def _states(n, seed, device, narrow=False):
    """Chemistry states as a burning H2-air flow has them: a mixture fraction,
    a progress from fresh to burnt, radicals of every size, temperature rising
    with the progress, near-atmospheric pressure, time steps of the solver.
    Species order H2 H O2 O OH HO2 H2O2 H2O N2.  narrow: within the box that
    the mixing-layer surrogate is trusted on."""
    g = torch.Generator().manual_seed(seed)
    u = torch.rand(14, n, generator=g, dtype=torch.float64)
    z = 0.002 + 0.1 * u[0] ** 2
    h2, o2 = z, 0.233 * (1 - z)
    burn = u[1] * torch.minimum(h2, o2 / 8)
    y = torch.zeros(9, n, dtype=torch.float64)
    y[0], y[2], y[7], y[8] = h2 - burn, o2 - 8 * burn, 9 * burn, 0.767 * (1 - z)
    for q, k in enumerate((1, 3, 4, 5, 6)):
        y[k] = 10.0 ** (-13 + 7.5 * u[2 + q])
    y /= y.sum(0)
    t = 1000 + 300 * u[7] + 1000 * burn / torch.minimum(h2, o2 / 8) * (0.3 + 0.5 * u[8])
    t, p = (t.clamp(980, 2180), 101325 * (0.95 + 0.1 * u[9])) if narrow else (t + 300 * u[9], 101325 * (0.6 + 2 * u[10]))
    dt = 10.0 ** (-7.8 + 0.6 * u[11])
    return [a.contiguous().to(device) for a in (t, p, y.t(), dt)]


def _targets(n, seed, device):
    g = torch.Generator().manual_seed(seed + 7)
    o = torch.zeros(n, 16, dtype=torch.float32)
    o[:, :10] = torch.randn(n, 10, generator=g)
    return o.to(device)


def _chemistry_context():
    mech, _ = workloads.load_mechanism(True)
    y = np.zeros(mech.n_spec)
    y[2], y[8] = 0.233, 0.767
    air = workloads.mixture_inflow(mech, y, 2.0, 101325.0, 1500.0)
    return Context(workloads.mixture_param(mech, False, True, 4, 0.2, 1, air))


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("box", "plate", "mixing", "jet"):
        flow = _flow_case(case, seed)
        sim = Simulation(flow)
        for blk in flow.blocks:  # the device holds them now
            blk.xg = blk.yg = blk.zg = blk.jac = blk.metric = blk.bv0 = blk.sv0 = None
        sim.initialize_computation()
        rans = flow.param.turb_method == L.RANS
        views = []
        for zone in sim.zones:
            sv = _interior(zone, "SV") if flow.param.n_scalar else None
            views.append(_fields(flow.param, _interior(zone, "BV"), sv, _interior(zone, "CV"),
                                 _interior(zone, "MUL")[0], _interior(zone, "LAMBDA")[0],
                                 _interior(zone, "MUT")[0] if rans else None))
        return dict(kind=kind, sim=sim, views=views)
    ctx = _chemistry_context()
    n = case["n"]
    t, p, y, dt = _states(n, seed, "cuda", case.get("weights") == "hswish")
    s = dict(kind=kind, ctx=ctx, n=n, arrays=(t, p, y, dt), ptr=[C.c_void_p(a.data_ptr()) for a in (t, p, y, dt)])
    if kind in ("chemistry", "surrogate"):
        s["out"] = torch.zeros(n, 9, dtype=torch.float64, device="cuda")
    if kind == "surrogate":
        s["net"] = sur.Surrogate.load(ctx, WEIGHTS[case["weights"]])
    if kind == "gradients":
        s["net"] = sur.Surrogate.load(ctx, WEIGHTS[case["weights"]], max_batch=n)
        s["target"] = _targets(n, seed, "cuda")
        s["out"] = torch.zeros(s["net"].n_params, dtype=torch.float32, device="cuda")
    return s


def run(state):
    kind = state["kind"]
    if "sim" in state:
        state["sim"].step(NO_RESIDUAL)
        return state["views"]
    out = C.c_void_p(state["out"].data_ptr())
    if kind == "chemistry":
        ctx = state["ctx"]
        L.check(ctx.lib.ostc_chem_plain_step(ctx.h, state["n"], *state["ptr"], out, None), "chemistry step")
    elif kind == "surrogate":
        state["net"].step(state["n"], *state["ptr"], out)
    else:
        loss = state["net"].gradients(state["n"], *state["ptr"], None, C.c_void_p(state["target"].data_ptr()), out)
        return dict(gradients=state["out"], loss=loss)
    return state["out"]


def work(case):
    """Each input read once and each output written once; operations by a count
    of the formulas per cell (transcendentals as one)."""
    kind = case["kind"]
    if kind == "chemistry":
        return dict(bytes=case["n"] * 8 * (12 + 9), flops=case["n"] * 3174)
    if kind == "surrogate":
        return dict(bytes=case["n"] * 8 * (12 + 9), flops=case["n"] * 2 * (12 * 128 + 3 * 128 * 128 + 128 * 10))
    if kind == "gradients":
        params = 12 * 128 + 3 * 128 * 128 + 128 * 10
        return dict(bytes=case["n"] * (8 * 12 + 4 * 16) + 4 * params, flops=case["n"] * 6 * params)
    cells = case["mx"] * case["my"] * case["mz"] * (case["blocks"] if kind == "jet" else 1)
    ns, nt = {"box": (0, 0), "plate": (0, 2), "mixing": (9, 0), "jet": (9, 2)}[kind]
    nv, sweeps = 5 + ns + nt, case.get("steps", 0)
    # read: bv, scalars, cv, metric, Jacobian, wall distance; written: bv, scalars, cv
    scalars = 2 * (6 + ns + nt + nv) + 10 + (1 if nt else 0)
    face = 60 + 14 * nv + (40 * ns if ns else 10) + (0 if kind == "box" else 150 + 25 * (ns + nt))
    flops = 3 * face + sweeps * 3 * 10 * nv + 20 * nv + (150 if nt else 0) + (9 * 9 * 12 if ns else 10)
    if kind == "jet" or case.get("reacting"):
        flops += 3174 + sweeps * 2 * 81
    return dict(bytes=cells * scalars * case["precision"], flops=cells * flops)


def tolerance(case):
    """About four times the distance measured from the float64 statement.
    float32 flow: 3e-7 in the 2-norm (storage of the state); single points
    differ more where the T-from-e iteration, stopped at 1e-3, takes one pass
    more or less.  float64 flow and chemistry: 1e-15, and 2e-11 in a mixture,
    again from that iteration.  The network runs in bfloat16: a float32 sum next
    to a rounding boundary moves a hidden activation by one of its units (3e-3
    in the decoded changes, 2e-5 in the gradients of a whole batch)."""
    kind = case["kind"]
    if kind == "chemistry":
        return dict(rel=1e-12, max=1e-9)
    if kind == "surrogate":
        return dict(rel=1.5e-2, max=0.5)
    if kind == "gradients":
        return dict(rel=1e-4, max=5e-3)
    if case["precision"] == 8:
        return dict(rel=1e-12, max=1e-10) if kind in ("box", "plate") else dict(rel=1e-9, max=1e-5)
    return dict(rel=2e-6, max=2e-4)


# ------------------------------------------------------- the 64-bit statement

def exact(case, seed):
    kind = case["kind"]
    if kind in ("box", "plate", "mixing", "jet"):
        cells = case["mx"] * case["my"] * case["mz"] * (case["blocks"] if kind == "jet" else 1)
        if not torch.cuda.is_available() and cells > 200000:
            return None  # over 20 seconds on the CPU
        return _Flow(_flow_case(case, seed)).iteration()
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    mech = _Mixture(workloads.load_mechanism(True)[0], dev)
    t, p, y, dt = _states(case["n"], seed, dev, case.get("weights") == "hswish")
    if kind == "chemistry":
        return torch.cat([mech.plain_step(*[a[q:q + 200000] for a in (t, p, y, dt)])
                          for q in range(0, case["n"], 200000)])
    net = _Network(WEIGHTS[case["weights"]], dev)
    if kind == "surrogate":
        dy = net.change(t, p, y, dt)
        plain = torch.cat([mech.plain_step(*[a[q:q + 200000] for a in (t, p, y, dt)])
                           for q in range(0, case["n"], 200000)])
        return torch.where(net.trusted(t, p, y, dt, dy)[:, None], dy, plain)
    return net.gradients(t, p, y, dt, _targets(case["n"], seed, dev))


def _bf16(x):
    """x as bfloat16 holds it; derivatives pass through."""
    return x + (x.detach().float().bfloat16().double() - x.detach())


class _Network:
    """The surrogate: 12 features, four hidden layers of 128, standardised.  It
    is defined with bfloat16 features, weights and hidden activations; its sums
    and everything else are 64-bit here."""

    def __init__(self, path, dev):
        m = np.load(path, allow_pickle=False)
        self.d = {k[5:]: torch.as_tensor(np.asarray(m[k], np.float64), device=dev) for k in m.files
                  if k.startswith("desc_")}
        self.n_out = int(self.d["n_out"])
        self.act = int(self.d["activation"]) if "activation" in self.d else 0
        w = torch.as_tensor(m["weights"].astype(np.float64), device=dev)
        self.layers, at = [], 0
        for q in range(5):
            fin, fout = 12 if q == 0 else 128, self.n_out if q == 4 else 128
            self.layers.append([w[at:at + fin * fout].reshape(fout, fin), w[at + fin * fout:at + (fin + 1) * fout]])
            at += (fin + 1) * fout

    def outputs(self, t, p, y, dt):
        f = torch.cat([(1000 / t)[:, None], torch.log(p / 101325)[:, None], (y.clamp(min=0) ** 0.1 - 1) * 10,
                       torch.log(dt)[:, None]], 1)
        x = (f - self.d["in_mean"]) / self.d["in_std"]
        for q, (w, b) in enumerate(self.layers):
            x = torch.addmm(b, _bf16(x), _bf16(w).t())
            if q < 4:
                x = torch.nn.functional.gelu(x, approximate="tanh") if self.act == 0 else \
                    x * (x / 6 + 0.5).clamp(0, 1)
        return x

    def change(self, t, p, y, dt):
        o = torch.cat([self.outputs(*[a[q:q + 200000] for a in (t, p, y, dt)]) for q in range(0, len(t), 200000)])
        o = o * self.d["out_std"][:self.n_out] + self.d["out_mean"][:self.n_out]
        return o[:, 1:10] * 10 ** o[:, :1] if int(self.d["kind"]) == 0 else self.d["floor"] * torch.sinh(o[:, :9])

    def trusted(self, t, p, y, dt, dy):
        d = self.d
        ok = (t >= d["t_min"]) & (t <= d["t_max"]) & (p >= d["p_min"]) & (p <= d["p_max"])
        ok &= (dt >= d["dt_min"]) & (dt <= d["dt_max"]) & (y >= -d["y_tol"]).all(1)
        yn = y + dy
        ok &= ((yn >= -d["y_tol"]) & (yn <= 1 + d["y_tol"])).all(1)
        if "dy_max" in d:
            ok &= (dy.abs() <= d["dy_max"]).all(1)
        q = dy[:, None, :] * d["elem_w"].reshape(-1, 9)[:int(d["n_elem"])]
        return ok & (q.sum(2).abs().amax(1) <= d["elem_tol"] * q.abs().sum((1, 2)) + d["elem_abs"])

    def gradients(self, t, p, y, dt, target):
        leaves = [a.clone().requires_grad_() for layer in self.layers for a in layer]
        self.layers = [[leaves[2 * q], leaves[2 * q + 1]] for q in range(5)]
        diff = self.outputs(t, p, y, dt) - target[:, :self.n_out].double()
        loss = (self.d["loss_w"][:self.n_out] * diff ** 2).sum() / len(t)
        grads = torch.autograd.grad(loss, leaves)
        return dict(gradients=torch.cat([g.reshape(-1) for g in grads]), loss=float(loss))


RU, RC, P_ATM, MW_AIR, GAMMA_AIR = 8314.462618, 1.98720425864083, 101325.0, 28.9647, 1.4


class _Mixture:
    """Thermodynamics, transport and kinetics; species along the first axis."""

    def __init__(self, param, dev):
        ns, st = param.n_spec, L.MAX_SPEC
        self.ns, self.nr = ns, param.n_reac

        def t(a):
            return torch.tensor(list(a), dtype=torch.float64, device=dev)

        self.mw, self.t_low, self.t_mid = t(param.mw)[:ns], t(param.t_low)[:ns], t(param.t_mid)[:ns]
        self.low = t(param.low_temp_coeff).reshape(-1, 7)[:ns]
        self.high = t(param.high_temp_coeff).reshape(-1, 7)[:ns]
        self.lj, self.vis = t(param.LJ_potent_inv)[:ns], t(param.vis_coeff)[:ns]
        self.w14 = t(param.WjDivWi_to_One4th).reshape(st, st)[:ns, :ns]
        self.w8 = t(param.sqrt_WiDivWjPl1Mul8).reshape(st, st)[:ns, :ns]
        self.sc = param.Sc
        self.nu_f = t(param.stoi_f).reshape(-1, st)[:self.nr, :ns]
        self.nu_b = t(param.stoi_b).reshape(-1, st)[:self.nr, :ns]
        self.third = t(param.third_body_coeff).reshape(-1, st)[:self.nr, :ns]
        self.p = param

    def col(self, a, like):
        return a.reshape((-1,) + (1,) * like.dim())

    def coeffs(self, t):
        tl = torch.maximum(t[None], self.col(self.t_low, t))
        hot = tl >= self.col(self.t_mid, t)
        return tl, [torch.where(hot, self.col(self.high[:, q], t), self.col(self.low[:, q], t)) for q in range(7)]

    def h_cp(self, t):
        tl, a = self.coeffs(t)
        cp = a[0] + tl * (a[1] + tl * (a[2] + tl * (a[3] + tl * a[4])))
        h = a[5] + tl * (a[0] + tl * (a[1] / 2 + tl * (a[2] / 3 + tl * (a[3] / 4 + tl * a[4] / 5))))
        r = self.col(RU / self.mw, t)
        return (h + cp * (t[None] - tl)) * r, cp * r

    def gibbs(self, t):
        tl, a = self.coeffs(t)
        h = a[0] + a[5] / tl + tl * (a[1] / 2 + tl * (a[2] / 3 + tl * (a[3] / 4 + tl * a[4] / 5)))
        s = a[0] * torch.log(tl) + a[6] + tl * (a[1] + tl * (a[2] / 2 + tl * (a[3] / 3 + tl * a[4] / 4)))
        return h - s

    def mean_mw(self, y):
        return 1 / (y / self.col(self.mw, y[0])).sum(0)

    def transport(self, t, y, cp):
        mw = self.mean_mw(y)
        x = y * mw / self.col(self.mw, t)
        td = t[None] * self.col(self.lj, t)
        vis = self.col(self.vis, t) * torch.sqrt(t) / (1.147 * td ** -0.145 + (td + 0.5) ** -2)
        mu, lam = torch.zeros_like(t), torch.zeros_like(t)
        for m in range(self.ns):
            s = torch.zeros_like(t)
            for n in range(self.ns):
                phi = 1.0 if m == n else (1 + torch.sqrt(vis[m] / vis[n]) * self.w14[m, n]) ** 2 * self.w8[m, n]
                s += phi * x[n]
            mu += vis[m] * x[m] / s
            if cp is not None:
                lam += vis[m] * (cp[m] + 1.25 * RU / self.mw[m]) * x[m] / (1.065 * s - 0.065 * x[m])
        rho_d = torch.where((x - 1).abs() < 1e-3, mu / self.sc, (1 - y) * mu / ((1 - x) * self.sc))
        return mu, lam, rho_d

    def rates(self, rho, t, y):
        """Production rates and their Jacobian with frozen rate constants."""
        p, ns = self.p, self.ns
        c = rho * y / self.col(self.mw, t) * 1e-3
        g, lt = self.gibbs(t), torch.log(t)
        base = P_ATM / RU * 1e-3 / t

        def arr(a, b, e):
            return a * torch.exp(b * lt - e / t)

        omega = torch.zeros_like(y)
        jac = torch.zeros((ns, ns) + tuple(t.shape), dtype=torch.float64, device=t.device)
        for r in range(self.nr):
            kind, nf, nb = p.reac_type[r], self.nu_f[r].tolist(), self.nu_b[r].tolist()
            kf = arr(p.A[r], p.b[r], p.Ea[r])
            if kind == 3:
                kf = kf + arr(p.A2[r], p.b2[r], p.Ea2[r])
            elif kind > 3:
                cc = (c * self.col(self.third[r], t)).sum(0)
                if kind == 4:
                    kf = kf * cc
                else:
                    pr = arr(p.A2[r], p.b2[r], p.Ea2[r]) * cc / kf
                    f = 1.0
                    if kind > 5:
                        al = p.troe_alpha[r]
                        fc = (1 - al) * torch.exp(-t / p.troe_t3[r]) + al * torch.exp(-t / p.troe_t1[r])
                        if kind == 7:
                            fc = fc + torch.exp(-p.troe_t2[r] / t)
                        lf, lp = torch.log10(fc), torch.log10(pr)
                        c1, nn = -0.4 - 0.67 * lf, 0.75 - 1.27 * lf
                        f = 10 ** (lf / (1 + ((lp + c1) / (nn - 0.14 * (lp + c1))) ** 2))
                    kf = kf * pr / (1 + pr) * f
            if kind == 2:
                kb = arr(p.A2[r], p.b2[r], p.Ea2[r])
            else:
                dg = sum(g[k] * (nb[k] - nf[k]) for k in range(ns) if nb[k] or nf[k])
                kb = kf * torch.exp(dg) * base ** (-p.reac_order[r])
            for k in range(ns):
                kf = kf * c[k] ** int(nf[k]) if nf[k] else kf
                kb = kb * c[k] ** int(nb[k]) if nb[k] else kb
            for m in range(ns):
                d = nb[m] - nf[m]
                if not d:
                    continue
                omega[m] += d * (kf - kb)
                for n in range(ns):
                    if nf[n] or nb[n]:
                        jac[m, n] += d * (nf[n] * kf - nb[n] * kb)
        omega *= self.col(self.mw, t) * 1e3
        on = y > 1e-25
        scale = torch.where(on, 1 / (rho * torch.where(on, y, torch.ones_like(y))), torch.zeros_like(y))
        for m in range(ns):
            jac[m] *= scale * self.mw[m] * 1e3
        return omega, jac

    def plain_step(self, t, p, y, dt):
        y = y.t().contiguous()
        rho = p * self.mean_mw(y) / (RU * t)
        omega, jac = self.rates(rho, t, y)
        block = _Block(jac * (-dt), torch.ones_like(t))
        return (block.solve(omega * dt) / rho).t()

    def temperature(self, t, y, e):
        """The solver's Newton iteration, stopped where it stops."""
        gas = (y * self.col(RU / self.mw, t)).sum(0)
        left = torch.ones_like(t, dtype=torch.bool)
        for _ in range(60):
            h, cp = self.h_cp(t)
            new = t - ((h * y).sum(0) - gas * t - e) / ((cp * y).sum(0) - gas)
            err = (1 - new / t).abs()
            t = torch.where(left, new, t)
            left = left & (err > 1e-3)
            if not bool(left.any()):
                break
        return t, gas


class _Block:
    """LU factors of matrices a + diag I, one per point (first two axes)."""

    def __init__(self, a, diag):
        n = a.shape[0]
        for q in range(n):
            a[q, q] += diag
        for k in range(n):
            for m in range(k + 1, n):
                a[m, k] /= a[k, k]
                a[m, k + 1:] -= a[m, k] * a[k, k + 1:]
        self.a = a

    def solve(self, b):
        a, x = self.a, b.clone()
        n = a.shape[0]
        for m in range(1, n):
            x[m] -= (a[m, :m] * x[:m]).sum(0)
        for m in range(n - 1, -1, -1):
            if m < n - 1:
                x[m] -= (a[m, m + 1:] * x[m + 1:]).sum(0)
            x[m] /= a[m, m]
        return x


SK = dict(sk1=0.85, sk2=1.0, so1=0.5, so2=0.856, b1=0.075, b2=0.0828, bs=0.09, a1=0.31)
SK["g1"] = SK["b1"] / SK["bs"] - SK["so1"] * 0.41 ** 2 / 0.3
SK["g2"] = SK["b2"] / SK["bs"] - SK["so2"] * 0.41 ** 2 / 0.3


def _sutherland(t):
    return 1.716e-5 * (t / 273) ** 1.5 * 384 / (t + 111)


class _Zone:
    pass


class _Flow:
    """One steady iteration on padded blocks [variable, k, j, i], g = 2."""

    def __init__(self, case):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.case, self.p, self.g = case, case.param, case.ngg
        p = case.param
        self.ns = p.n_spec
        self.nt = 2 if p.turb_method == L.RANS else 0
        self.mix = _Mixture(p, self.dev) if self.ns else None
        self.reacting = p.mix_model == L.FR
        self.zones = [self.zone(b) for b in case.blocks]

    def load(self, a):
        t = torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64), device=self.dev)
        return t.float().double() if self.case.precision == 4 else t

    def zone(self, blk):
        z = _Zone()
        z.blk, z.m = blk, (blk.mx, blk.my, blk.mz)
        z.metric = self.load(blk.metric).reshape((3, 3) + blk.jac.shape)
        z.jac = self.load(blk.jac)
        z.bv = self.load(blk.bv0).clone()
        z.sv = self.load(blk.sv0).clone() if self.p.n_scalar else z.bv[:0]
        zero = torch.zeros_like(z.jac)
        z.cv = zero.expand((self.p.n_var,) + zero.shape).clone()
        z.mut, z.lamt, z.wall = zero.clone(), zero.clone(), None
        if self.nt:
            xyz = [torch.as_tensor(np.ascontiguousarray(a), device=self.dev).reshape(-1)
                   for a in (blk.xg, blk.yg, blk.zg)]
            z.wall = self.load_t(self.distance(xyz).reshape(zero.shape))
        return z

    def load_t(self, t):
        return t.float().double() if self.case.precision == 4 else t

    def distance(self, xyz):
        wp = torch.as_tensor(np.ascontiguousarray(self.case.wall_points), device=self.dev)
        best = torch.full_like(xyz[0], 1e6)
        step = max(1, int(3e7) // len(wp))
        for q in range(0, len(best), step):
            d = sum((xyz[c][q:q + step, None] - wp[None, :, c]) ** 2 for c in range(3))
            best[q:q + step] = torch.minimum(best[q:q + step], d.amin(1))
        return torch.sqrt(best)

    # ---- points, with `lo`/`hi` more of them on both ends of each direction
    def box(self, z, a, lo=(0, 0, 0), hi=(0, 0, 0)):
        s = [slice(self.g + lo[d], self.g + z.m[d] + hi[d]) for d in (2, 1, 0)]
        return a[(Ellipsis, *s)]

    def shifted(self, z, a, d, s):
        off = [0, 0, 0]
        off[d] = s
        return self.box(z, a, off, off)

    # ---- state and properties
    def energy(self, z):
        rho, vel2 = z.bv[0], (z.bv[1:4] ** 2).sum(0)
        e = 0.5 * rho * vel2
        if self.ns:
            return e + (self.mix.h_cp(z.bv[5])[0] * z.sv[:self.ns]).sum(0) * rho - z.bv[4]
        return e + z.bv[4] / (GAMMA_AIR - 1)

    def conserved(self, z):
        z.cv = torch.cat([z.bv[:1], z.bv[0] * z.bv[1:4], self.energy(z)[None], z.bv[0] * z.sv])

    def properties(self, z):
        t = z.bv[5]
        if self.ns:
            h, cp = self.mix.h_cp(t)
            y = z.sv[:self.ns]
            gas = (y * self.mix.col(RU / self.mix.mw, t)).sum(0)
            z.cp = (cp * y).sum(0)
            z.gamma = z.cp / (z.cp - gas)
            z.sound = torch.sqrt(z.gamma * gas * t)
            z.mul, z.lam, z.rho_d = self.mix.transport(t, y, cp)
        else:
            z.cp = torch.full_like(t, GAMMA_AIR * RU / MW_AIR / (GAMMA_AIR - 1))
            z.gamma = torch.full_like(t, GAMMA_AIR)
            z.sound = torch.sqrt(GAMMA_AIR * RU / MW_AIR * t)
            z.mul = _sutherland(t)
            z.lam = z.mul * z.cp / self.p.Pr

    def grad(self, z, f, one=0):
        """Central gradient of f at the interior points (`one` more around)."""
        n = (one, one, one)
        lo, out = tuple(-o for o in n), []
        d = []
        for q in range(3):
            up, dn = list(n), list(lo)
            a, b = list(lo), list(n)
            a[q] += 1
            b[q] += 1
            hi = self.box(z, f, a, b)
            a[q] -= 2
            b[q] -= 2
            d.append(0.5 * (hi - self.box(z, f, a, b)))
        m = self.box(z, z.metric, lo, n)
        return [m[0, c] * d[0] + m[1, c] * d[1] + m[2, c] * d[2] for c in range(3)]

    def eddy(self, z, u, v, w, rho, k, om, rho_k, mul, dy):
        vort = torch.sqrt((v[0] - u[1]) ** 2 + (w[0] - u[2]) ** 2 + (w[1] - v[2]) ** 2)
        ok = dy > 1e-25
        d = torch.where(ok, dy, torch.ones_like(dy))
        arg = torch.maximum(2 * torch.sqrt(k) / (0.09 * om * d), 500 * mul / (rho * d * d * om))
        f2 = torch.where(ok, torch.tanh(arg ** 2), torch.ones_like(dy))
        den = torch.maximum(SK["a1"] * om, vort * f2)
        return torch.where(den > 1e-25, SK["a1"] * rho_k / den, torch.zeros_like(den))

    def initial_eddy(self, z):
        n = (1, 1, 1)
        lo = (-1, -1, -1)
        at = lambda a: self.box(z, a, lo, n)  # noqa: E731
        u, v, w = (self.grad(z, z.bv[q], 1) for q in (1, 2, 3))
        mul = self.mix.transport(at(z.bv[5]), at(z.sv[:self.ns]), None)[0] if self.ns else _sutherland(at(z.bv[5]))
        k, om = at(z.sv[self.ns]), at(z.sv[self.ns + 1])
        at(z.mut)[...] = self.eddy(z, u, v, w, at(z.bv[0]), k, om, at(z.cv[5 + self.ns]), mul, at(z.wall))

    # ---- boundaries
    def face_points(self, f, shift):
        s = [slice(self.g + f.range_start[q], self.g + f.range_end[q] + 1) for q in range(3)]
        a = self.g + f.range_start[f.face] + shift * f.direction
        s[f.face] = slice(a, a + 1)
        return (Ellipsis, s[2], s[1], s[0])

    def boundaries(self, z):
        bc, g = z.blk.bc, self.g
        for q in range(bc.n_face):
            f = bc.face[q]
            at = [self.face_points(f, s) for s in range(-g, g + 1)]  # at[g + s]
            if f.kind == 6:
                for s in range(1, g + 1):
                    for a in (z.bv, z.sv, z.mut):
                        a[at[g + s]] = a[at[g]]
            elif f.kind == 5:
                i = bc.inflow[f.slot]
                for s in range(1, g + 1):
                    for l, v in enumerate((i.density, i.u, i.v, i.w, i.pressure, i.temperature)):
                        z.bv[l][at[g + s]] = v
                    for l in range(self.p.n_scalar):
                        z.sv[l][at[g + s]] = i.sv[l]
                    z.mut[at[g + s]] = i.mut
            elif f.kind == 3:
                self.symmetry(z, f, at)
            else:
                self.wall(z, f, at, bc.wall[f.slot])

    def symmetry(self, z, f, at):
        g = self.g
        n = z.metric[f.face][at[g]]
        n = n / torch.sqrt((n ** 2).sum(0))
        new = []
        for s in range(0, g + 1):
            src = at[g - max(s, 1)]
            bv, sv, mut = z.bv[src].clone(), z.sv[src].clone(), z.mut[src].clone()
            old = bv[1:4].clone()
            bv[1:4] -= (1 if s == 0 else 2) * (n * old).sum(0) * n
            new.append((s, bv, sv, mut, old))
        e1 = z.cv[4][at[g - 1]].clone()
        for s, bv, sv, mut, old in new:
            z.bv[at[g + s]], z.sv[at[g + s]] = bv, sv
            if s:
                z.mut[at[g + s]] = mut
                continue
            e = e1 - 0.5 * bv[0] * (old ** 2).sum(0) + 0.5 * bv[0] * (bv[1:4] ** 2).sum(0)
            z.cv[at[g]] = torch.cat([bv[:1], bv[0] * bv[1:4], e[None], bv[0] * sv])

    def wall(self, z, f, at, wall):
        g, ns = self.g, self.ns
        bv1, sv1 = z.bv[at[g - 1]].clone(), z.sv[at[g - 1]].clone()
        y = sv1[:ns]
        tw = torch.full_like(bv1[5], wall.temperature) if wall.isothermal else bv1[5]
        mw = self.mix.mean_mw(y) if ns else MW_AIR
        rho = bv1[4] * mw / (tw * RU)
        om = None
        if self.nt:
            mu = self.mix.transport(tw, y, None)[0] if ns else _sutherland(tw)
            dy = z.wall[at[g - 1]]
            ok = dy > 1e-25
            om = torch.where(ok, 60 * mu / (rho * SK["b1"] * torch.where(ok, dy, torch.ones_like(dy)) ** 2), sv1[ns + 1])
        ghosts = [(s, z.bv[at[g - s]].clone(), z.sv[at[g - s]].clone()) for s in range(1, g + 1)]
        zero = torch.zeros_like(rho)
        turb = torch.stack([zero, om]) if self.nt else sv1[ns:]
        z.bv[at[g]] = torch.stack([rho, zero, zero, zero, bv1[4], tw])
        z.sv[at[g]] = torch.cat([y, turb])
        e = (self.mix.h_cp(tw)[0] * y).sum(0) * rho - bv1[4] if ns else bv1[4] / (GAMMA_AIR - 1)
        z.cv[at[g]] = torch.cat([torch.stack([rho, zero, zero, zero, e]), rho * z.sv[at[g]]])
        for s, bv, sv in ghosts:
            t = bv[5]
            if wall.isothermal:
                t = 2 * tw - bv[5]
                t = torch.where(t <= 0.1 * tw, tw, t)
            m = self.mix.mean_mw(sv[:ns]) if ns else MW_AIR
            z.bv[at[g + s]] = torch.cat([(bv[4] * m / (t * RU))[None], -bv[1:4], bv[4:5], t[None]])
            z.sv[at[g + s]] = torch.cat([sv[:ns], turb])
            z.mut[at[g + s]] = 0

    def primitives(self, cv, t):
        rho, vel = cv[0], cv[1:4] / cv[0]
        sv, vel2 = cv[5:] / rho, (vel ** 2).sum(0)
        if self.ns:
            t, gas = self.mix.temperature(t, sv[:self.ns], cv[4] / rho - 0.5 * vel2)
            p = rho * t * gas
        else:
            p = (GAMMA_AIR - 1) * (cv[4] - 0.5 * rho * vel2)
            t = p * MW_AIR / (rho * RU)
        return torch.cat([rho[None], vel, p[None], t[None]]), sv

    def exchange(self):
        g = self.g
        for z in self.zones:
            for f in z.blk.inner:
                t = self.zones[f.target_block]
                n = torch.meshgrid(*[torch.arange(f.n_point[q], device=self.dev) for q in (0, 1, 2)], indexing="ij")
                d = [f.loop_dir[q] * n[q] for q in range(3)]
                a = [f.range_start[q] + d[q] for q in range(3)]
                b = [f.target_start[q] + f.target_loop_dir[q] * d[f.src_tar[q]] for q in range(3)]
                on = a[f.face] == (f.range_start[f.face] if f.direction > 0 else f.range_end[f.face])
                pick = lambda i, m: tuple((i[q] + g)[m] for q in (2, 1, 0))  # noqa: E731
                ia, ib = (slice(None),) + pick(a, on), (slice(None),) + pick(b, on)
                ave = 0.5 * (t.cv[ib] + z.cv[ia])
                z.cv[ia] = ave
                t.cv[ib] = ave
                z.bv[ia], z.sv[ia] = self.primitives(ave, z.bv[5][ia[1:]])
                ia, ib = (slice(None),) + pick(a, ~on), (slice(None),) + pick(b, ~on)
                z.bv[ia], z.sv[ia] = t.bv[ib], t.sv[ib]

    # ---- one iteration
    def iteration(self):
        for z in self.zones:
            self.boundaries(z)
        for z in self.zones:
            self.conserved(z)
            if self.nt:
                self.initial_eddy(z)
        self.exchange()
        for z in self.zones:
            self.properties(z)
        for z in self.zones:
            self.advance(z)
        self.exchange()
        out = []
        for z in self.zones:
            self.properties(z)
            mut = self.box(z, z.mut) if self.nt else None
            out.append(_fields(self.p, self.box(z, z.bv), self.box(z, z.sv), self.box(z, z.cv), self.box(z, z.mul),
                               self.box(z, z.lam), mut))
        return out

    def advance(self, z):
        p, ns, nt = self.p, self.ns, self.nt
        at = lambda a: self.box(z, a)  # noqa: E731
        jac, rho, vel, m = at(z.jac), at(z.bv[0]), at(z.bv[1:4]), at(z.metric)
        rhs = torch.zeros((p.n_var,) + jac.shape, dtype=torch.float64, device=self.dev)
        tj = block = None
        if nt:
            tj = self.turbulence(z, rhs)
        if self.reacting:
            omega, cj = self.mix.rates(rho, at(z.bv[5]), at(z.sv[:ns]))
            rhs[5:5 + ns] = jac * omega
        for d in range(3):
            flux = self.inviscid(z, d)
            if p.viscous_scheme:
                flux -= self.viscous(z, d)
            ax = 3 - d
            n = z.m[d]
            rhs -= flux.narrow(ax, 1, n) - flux.narrow(ax, 0, n)
            del flux
        # local time step
        size = torch.sqrt((m ** 2).sum(1))
        radius = (m * vel[None]).sum(1).abs() + at(z.sound) * size
        visc = at(z.mul) / p.Pr + (at(z.mut) / p.Prt if nt else 0)
        srv = (size ** 2).sum(0) * torch.clamp(at(z.gamma), min=4 / 3) / rho * visc
        dt = p.cfl / (radius.sum(0) + srv)
        dq = rhs
        if p.implicit_method == 1:
            diag = 1 + dt * radius.sum(0)
            if self.reacting:
                block = _Block(cj.mul_(-dt), diag)

            def scale(r):
                out = r / diag
                if block is not None:
                    out[5:5 + ns] = block.solve(r[5:5 + ns])
                if nt:
                    for q in range(2):
                        out[5 + ns + q] = r[5 + ns + q] / (diag - dt * tj[q])
                return out

            dq0 = scale(rhs)
            dq = dq0
            for _ in range(p.dplur_inner_step):
                dq = dq0 + scale(dt * self.neighbours(z, dq, radius))
        cv = at(z.cv)
        cv += dq * dt / jac
        bv, sv = self.primitives(cv, at(z.bv[5]))
        at(z.bv)[...] = bv
        at(z.sv)[...] = sv
        self.boundaries(z)

    def turbulence(self, z, rhs):
        ns = self.ns
        at = lambda a: self.box(z, a)  # noqa: E731
        u, v, w = (self.grad(z, z.bv[q]) for q in (1, 2, 3))
        gk, go = self.grad(z, z.sv[ns]), self.grad(z, z.sv[ns + 1])
        rho, k, om, mul, dy = at(z.bv[0]), at(z.sv[ns]), at(z.sv[ns + 1]), at(z.mul), at(z.wall)
        inter = 2 * rho * SK["so2"] / om * sum(gk[c] * go[c] for c in range(3))
        mut = self.eddy(z, u, v, w, rho, k, om, rho * k, mul, dy)
        f1 = self.blend(rho, k, om, mul, dy, inter)
        at(z.mut)[...] = mut
        at(z.lamt)[...] = mut * at(z.cp) / self.p.Prt
        beta = SK["b2"] + (SK["b1"] - SK["b2"]) * f1
        div = u[0] + v[1] + w[2]
        prod = mut * (2 * (u[0] ** 2 + v[1] ** 2 + w[2] ** 2) - 2 / 3 * div ** 2 + (u[1] + v[0]) ** 2 +
                      (u[2] + w[0]) ** 2 + (v[2] + w[1]) ** 2) - 2 / 3 * rho * k * div
        on = mut > 1e-25
        safe = torch.where(on, mut, torch.ones_like(mut))
        gam = SK["g2"] + (SK["g1"] - SK["g2"]) * f1
        zero = torch.zeros_like(mut)
        rhs[5 + ns] = torch.where(on, at(z.jac) * (prod - SK["bs"] * rho * k * om), zero)
        rhs[6 + ns] = torch.where(on, at(z.jac) * (gam * rho / safe * prod + (1 - f1) * inter - beta * rho * om ** 2),
                                  zero)
        return -2 * SK["bs"] * om, -2 * beta * om

    def blend(self, rho, k, om, mul, dy, inter):
        ok = dy > 1e-25
        d = torch.where(ok, dy, torch.ones_like(dy))
        a1, a2 = torch.sqrt(k) / (0.09 * om * d), 500 * mul / (rho * d * d * om)
        a3 = 4 * rho * SK["so2"] * k / (torch.clamp(inter, min=1e-20) * d * d)
        return torch.where(ok, torch.tanh(torch.minimum(torch.maximum(a1, a2), a3) ** 4), torch.ones_like(dy))

    def faces(self, z, a, d, s, e=None, t=0):
        """Values at point f - 1 + s of every face f = 0 .. n along d, moved by t along e."""
        lo, hi = [0, 0, 0], [0, 0, 0]
        lo[d], hi[d] = s - 1, s
        if e is not None:
            lo[e] += t
            hi[e] += t
        return self.box(z, a, lo, hi)

    def area(self, z, d):
        l, r = self.faces(z, z.jac, d, 0), self.faces(z, z.jac, d, 1)
        return 0.5 * (self.faces(z, z.metric[d], d, 0) * l + self.faces(z, z.metric[d], d, 1) * r)

    def inviscid(self, z, d):
        ns = self.ns
        q = torch.cat([z.bv[:5], z.sv])
        pv = [self.faces(z, q, d, s) for s in (-1, 0, 1, 2)]

        def minmod(a, b):
            m = torch.minimum(a.abs(), b.abs())
            return torch.where((a < 0) == (b < 0), torch.where(a < 0, -m, m), torch.zeros_like(m))

        mid = pv[2] - pv[1]
        side = [pv[1] + 0.5 * minmod(pv[1] - pv[0], mid), pv[2] - 0.5 * minmod(mid, pv[3] - pv[2])]
        k = self.area(z, d)
        gk = torch.sqrt((k ** 2).sum(0))
        total, un, c = [], [], 0
        for s in side:
            ke = 0.5 * (s[1:4] ** 2).sum(0)
            if ns:
                y = s[5:5 + ns]
                gas = (y * self.mix.col(RU / self.mix.mw, s[0])).sum(0)
                h, cp = self.mix.h_cp(s[4] / (s[0] * gas))
                e, cpm = s[0] * (ke + (h * y).sum(0)) - s[4], (cp * y).sum(0)
                gam = cpm / (cp * y - y * self.mix.col(RU / self.mix.mw, s[0])).sum(0)
            else:
                e, gam = ke * s[0] + s[4] / (GAMMA_AIR - 1), GAMMA_AIR
            total.append((e + s[4]) / s[0])
            un.append((k * s[1:4]).sum(0) / gk)
            c = c + 0.5 * torch.sqrt(gam * s[4] / s[0])

        def split(mach, sign):
            sup, pol = 0.5 * (mach + sign * mach.abs()), 0.25 * (mach + sign) ** 2
            b = (mach * mach - 1) ** 2
            sub = sign * (pol + 0.125 * b)
            ps = pol * (2 - sign * mach) + sign * 3 / 16 * mach * b
            over = mach.abs() > 1
            safe = torch.where(over, mach, torch.ones_like(mach))
            return torch.where(over, sup, sub), torch.where(over, sup / safe, ps)

        (ml, pl), (mr, pr) = split(un[0] / c, 1), split(un[1] / c, -1)
        half = ml + mr
        flow = c * (side[0][0] * torch.clamp(half, min=0) + side[1][0] * torch.clamp(half, max=0))
        up = flow >= 0
        st = torch.where(up, side[0], side[1])
        flow = flow * gk
        press = (pl * side[0][4] + pr * side[1][4]) * k
        return torch.cat([flow[None], flow * st[1:4] + press, (flow * torch.where(up, *total))[None], flow * st[5:]])

    def viscous(self, z, d):
        p, ns, nt = self.p, self.ns, self.nt
        mean = lambda a: 0.5 * (self.faces(z, a, d, 0) + self.faces(z, a, d, 1))  # noqa: E731
        m, k = mean(z.metric), self.area(z, d)

        def grad(a):
            der = []
            for e in range(3):
                if e == d:
                    der.append(self.faces(z, a, d, 1) - self.faces(z, a, d, 0))
                else:
                    der.append(0.25 * sum(self.faces(z, a, d, s, e, 1) - self.faces(z, a, d, s, e, -1)
                                          for s in (0, 1)))
            return [m[0, c] * der[0] + m[1, c] * der[1] + m[2, c] * der[2] for c in range(3)]

        u = [grad(z.bv[q]) for q in (1, 2, 3)]
        mul, mut = mean(z.mul), mean(z.mut)
        vis, div = mul + mut, u[0][0] + u[1][1] + u[2][2]
        normal = -2 / 3 * mean(z.bv[0] * z.sv[ns]) if nt else 0
        out = torch.zeros((p.n_var,) + k[0].shape, dtype=torch.float64, device=self.dev)
        for a in range(3):
            for b in range(3):
                tau = vis * (u[a][b] + u[b][a])
                if a == b:
                    tau = tau - 2 / 3 * vis * div + normal
                out[1 + a] += k[b] * tau
        dt = grad(z.bv[5])
        cond = mean(z.lam) + (mean(z.lamt) if nt else 0)
        out[4] = (mean(z.bv[1:4]) * out[1:4]).sum(0) + cond * sum(k[c] * dt[c] for c in range(3))
        if ns:
            h = self.mix.h_cp(mean(z.bv[5]))[0]
            corr = 0
            for l in range(ns):
                g = grad(z.sv[l])
                dif = mean(z.rho_d[l]) + (mut / p.Sct if nt else 0)
                j = dif * sum(k[c] * g[c] for c in range(3))
                out[5 + l] = j
                out[4] += h[l] * j
                corr = corr + j
            for l in range(ns):
                out[5 + l] -= mean(z.sv[l]) * corr
        if nt:
            gk, go = grad(z.sv[ns]), grad(z.sv[ns + 1])
            rho, tk, om, dy = mean(z.bv[0]), mean(z.sv[ns]), mean(z.sv[ns + 1]), mean(z.wall)
            inter = 2 * rho * SK["so2"] / om * sum(gk[c] * go[c] for c in range(3))
            f1 = self.blend(rho, tk, om, mul, dy, inter)
            out[5 + ns] = (mul + mut * (SK["sk2"] + (SK["sk1"] - SK["sk2"]) * f1)) * sum(k[c] * gk[c] for c in range(3))
            out[6 + ns] = (mul + mut * (SK["so2"] + (SK["so1"] - SK["so2"]) * f1)) * sum(k[c] * go[c] for c in range(3))
        return out

    def neighbours(self, z, dq, radius):
        """Off-diagonal part of the split linearisation: what each cell takes
        from its six neighbours inside the block."""
        ns = self.ns
        at = lambda a: self.box(z, a)  # noqa: E731
        vel, t, gam, sv = at(z.bv[1:4]), at(z.bv[5]), at(z.gamma), at(z.sv)
        e = 0.5 * (vel ** 2).sum(0)
        b2 = (gam - 1) * (e * dq[0] - (vel * dq[1:4]).sum(0) + dq[4])
        if ns:
            h = self.mix.h_cp(t)[0]
            b2 = b2 + gam * t * (self.mix.col(RU / self.mix.mw, t) * dq[5:5 + ns]).sum(0)
            b2 = b2 - (gam - 1) * (h * dq[5:5 + ns]).sum(0)
            ht = (h * sv[:ns]).sum(0) + e
        else:
            ht = gam / (gam - 1) * at(z.bv[4]) / at(z.bv[0]) + e
        acc = torch.zeros_like(dq)
        for d in range(3):
            k = at(z.metric[d])
            un = (k * vel).sum(0)
            b1 = (k * dq[1:4]).sum(0) - un * dq[0]
            prod = torch.cat([(b1 + un * dq[0])[None], vel * b1 + k * b2 + un * dq[1:4],
                              (ht * b1 + un * b2 + un * dq[4])[None], un * dq[5:] + sv * b1])
            ax, n = 3 - d, z.m[d]
            plus, minus = 0.5 * (prod + radius[d] * dq), 0.5 * (prod - radius[d] * dq)
            acc.narrow(ax, 1, n - 1).add_(plus.narrow(ax, 0, n - 1))
            acc.narrow(ax, 0, n - 1).sub_(minus.narrow(ax, 1, n - 1))
        return acc
