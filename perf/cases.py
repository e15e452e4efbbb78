"""The work that performance is measured on: calls of the library's public entry points on
device-resident fields, as a model's time loop makes them.

Kinds of a case:

  step      one whole time step of the hot path through the fused entry points: ssh_nxt, wzv, step_dyn
            (dyn_adv, dyn_vor, dyn_spg_ts, dyn_zdf), div_hor, wzv, step_tra (tra_adv, tra_ldf_iso,
            tra_zdf), tra_nxt, dyn_nxt, ssh_swp
  routines  the same operators through the drop-in routines a model calls one by one: dyn_adv, dyn_vor,
            dyn_spg_ts, dyn_zdf, tra_adv_trp, tra_adv_fct, tra_ldf_lap, tra_zdf
  physics   the density, stratification, iso-neutral slopes, lateral viscosity and pressure gradient of
            a step: rab_3d, bn2, zdf_mxl, eos_insitu, ldf_slp, eos_insitu_pot, dyn_ldf_lap, hpg_zco
  adjoint   a tracer step and its gradient (nemo_hip.autograd): forward with the limiter's factors,
            backward with the factors frozen
  ensemble  one time step of several uneven domains, replayed from a plan

Grids: "gyre" is the closed flat-bottomed beta-plane basin, "basin" the seeded land mask with lognormal
bathymetry; a grid is fixed by its sizes (a program registers its domain once and keeps it), the fields
on it are drawn from the seed.  exact() repeats a pass in plain torch at 64 bits.
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "nemo-fmi-devel_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import nemo_hip  # noqa: E402
from nemo_hip import abi, autograd, configs  # noqa: E402

F64 = torch.float64
KT = 10                        # a leapfrog step, past the Euler start
ENSEMBLE_RANGE = ((128, 160), (384, 320))
GRID_SEED = 20261204
AHM, RN_SLPMAX, RHO_C = 2000.0, 0.01, 0.01


def _case(name, kind, jpi, jpj, jpk, dtype, **kw):
    c = dict(name=name, kind=kind, grid="basin", jpi=jpi, jpj=jpj, jpk=jpk, dtype=dtype, jperio=0, kn=4, vor="ene",
             eos="teos10", members=1)
    c.update(kw)
    return c


def listed():
    return [
        # the CPU-scale closed basin: a step is a long chain of very small launches
        _case("step_gyre_f64", "step", 32, 22, 31, "f64", grid="gyre", kn=2),
        # an ordinary regional domain, odd sizes, FP32 storage
        _case("step_regional_f32", "step", 251, 333, 56, "f32"),
        # an ordinary cyclic (channel) domain, FP64, the energy and enstrophy conserving vorticity
        _case("step_channel_f64", "step", 362, 149, 46, "f64", jperio=1, vor="een"),
        # the full-size domain in the FP32 storage form: the largest
        _case("step_full_f32", "step", 1024, 1024, 75, "f32"),
        # the plain FP64 form, routine by routine, as a model binds it
        _case("routines_f64", "routines", 512, 512, 75, "f64"),
        # ... and in FP32 storage on a small cyclic domain with second-order fluxes
        _case("routines_channel_f32", "routines", 182, 149, 31, "f32", jperio=1, kn=2, vor="een"),
        # density, slopes, viscosity and pressure gradient: TEOS-10 at 75 levels, FP32 storage
        _case("physics_f32", "physics", 512, 509, 75, "f32"),
        # ... simplified equation of state, FP64, small and cyclic
        _case("physics_channel_f64", "physics", 203, 157, 31, "f64", jperio=1, eos="seos"),
        # one step of a gradient of a tracer window
        _case("adjoint_f64", "adjoint", 256, 256, 75, "f64"),
        # a batch of uneven regional domains stepped together
        _case("ensemble_f32", "ensemble", 0, 0, 56, "f32", members=6),
    ]


def draw(rng):
    kind = rng.choice(["step", "step", "routines", "physics", "physics", "adjoint", "ensemble"])
    jpk = rng.randint(20, 80)
    if kind == "ensemble":
        return _drop(_case("", kind, rng.randint(1, 999), 0, jpk, rng.choice(["f64", "f32"]), kn=rng.choice([2, 4]),
                           members=rng.randint(2, 8)))
    cells = math.exp(rng.uniform(math.log(2.5e4), math.log(2.5e7)))
    aspect = math.exp(rng.uniform(-0.6, 0.6))
    side = math.sqrt(cells / jpk)
    jpi, jpj = max(20, int(side * aspect)), max(20, int(side / aspect))
    return _drop(_case("", kind, jpi, jpj, jpk, "f64" if kind == "adjoint" else rng.choice(["f64", "f32"]),
                       grid=rng.choice(["basin", "basin", "gyre"]), jperio=rng.choice([0, 0, 1]),
                       kn=rng.choice([2, 4]), vor=rng.choice(["ene", "een"]), eos=rng.choice(["teos10", "seos"])))


def _drop(c):
    del c["name"]
    return c


# ----------------------------------------------------------------------------
# grids, inputs and states
# ----------------------------------------------------------------------------
_GRIDS = {}                    # sizes and options -> (library context, domain); the domain is registered once
_GRID_CELLS = 400_000_000      # bound on the cells of the registered domains


def _members(case):
    """the grids of a case: one, or the uneven members of an ensemble"""
    if case["kind"] != "ensemble":
        return [case]
    import random
    r = random.Random(1000 * case["jpi"] + case["members"])
    (i0, j0), (i1, j1) = ENSEMBLE_RANGE
    return [dict(case, jpi=r.randint(i0, i1), jpj=r.randint(j0, j1)) for _ in range(case["members"])]


def _domain(g):
    opts = dict(nvor_scheme=abi.VOR_NAMES[g["vor"]], nn_baro=30, neuler=0, nit000=1)
    if g["grid"] == "gyre":
        return configs.gyre_like(g["jpi"], g["jpj"], g["jpk"], jperio=g["jperio"], opts=opts)
    return configs.basin(g["jpi"], g["jpj"], g["jpk"], seed=GRID_SEED + g["jpi"] + g["jpj"], jperio=g["jperio"],
                         opts=dict(opts, rdt=600.0))


def _grid(h, g):
    key = tuple(g[k] for k in ("grid", "jpi", "jpj", "jpk", "jperio", "vor", "eos"))
    if key not in _GRIDS:
        d = _domain(g)
        while _GRIDS and sum(k[1] * k[2] * k[3] for k in _GRIDS) + d.jpi * d.jpj * d.jpk > _GRID_CELLS:
            h.context_destroy(_GRIDS.pop(next(iter(_GRIDS)))[0])
        ctx = h.context_create()
        h.context_select(ctx)
        h.register(d)
        h.eos_register(abi.teos10() if g["eos"] == "teos10" else abi.seos())
        for n in abi.DOMAIN_3D_FIELDS:     # the library has its copies
            d.arrays[n] = None
        _GRIDS[key] = (ctx, d)
    return _GRIDS[key]


def _dt(case):
    return F64 if case["dtype"] == "f64" else torch.float32


THREED = ("un", "vn", "wn", "ub", "vb", "avt", "avm", "ahtu", "ahtv", "uslp", "vslp", "wslpi", "wslpj", "tsn", "tsb")


def _inputs(case, g, d, seed, device="cuda"):
    """The fields a step reads, drawn from the seed: 3D fields in the storage type, 2D ones in FP64."""
    S = configs.make_state_device(d, seed=seed, device=device)
    kind, dt = case["kind"], _dt(case)
    S.pop("tmask")
    S.pop("avs")
    if kind == "physics":
        S = {k: S[k] for k in ("tsn", "tsb", "ub", "vb", "un", "vn")}
    if kind == "adjoint":
        S = {k: S[k] for k in ("tsn", "tsb", "un", "vn", "wn", "ahtu", "ahtv", "avt")}
    X = {k: (v.to(dt) if k in THREED else v) for k, v in S.items()}
    gen = torch.Generator(device=device)
    gen.manual_seed(int(seed) + 17)
    n2, n3 = d.jpi * d.jpj, d.jpi * d.jpj * d.jpk
    if kind == "adjoint":
        X = {k: (v[:n3].clone() if k in ("tsn", "tsb") else v) for k, v in X.items()}
        X["gb"], X["gn"] = (torch.randn(n3, generator=gen, device=device, dtype=F64) for _ in range(2))
    elif kind == "physics":
        m = Masks(d, device)
        w, t = _depths(d, device)
        X["gdept"], X["gdepw"] = (_full(a, d).to(dt).reshape(-1) for a in (t, w))
        X["ahmt"], X["ahmf"] = ((AHM * a).to(dt).reshape(-1) for a in (m.t, m.f))
        X["ua"], X["va"] = 1e-6 * X.pop("un"), 1e-6 * X.pop("vn")     # trends of earlier operators
        # lateral density contrasts beside the vertical profile, so that the slopes are neither flat nor all capped
        y = torch.linspace(0.0, 1.0, d.jpj, device=device, dtype=F64)[None, :, None]
        x = torch.linspace(0.0, 1.0, d.jpi, device=device, dtype=F64)[None, None, :]
        for q in ("tsn", "tsb"):
            a = X[q].reshape(2, d.jpk, d.jpj, d.jpi)
            a[0] = ((a[0].double() - 3.0 * y - torch.sin(6.0 * x)) * m.t).to(dt)
            X[q] = a.reshape(-1)
    elif kind == "routines":
        X["ua"], X["va"] = 1e-6 * X["un"], 1e-6 * X["vn"]             # trends of earlier operators
        X["tsa"] = 1e-8 * X["tsn"]
    else:
        X["sshb"] = X["sshn"] * 0.99
        X["emp_b"] = X["emp"].clone()
    return X


def _full(a, d):
    return a[:, None, None].expand(d.jpk, d.jpj, d.jpi)


def _depths(d, device):
    """w- and t-point depths of the levels"""
    e3t, e3w = (torch.from_numpy(a).to(device) for a in (d.e3t_1d, d.e3w_1d))
    w = torch.cumsum(e3t, 0)
    return torch.cat([w.new_zeros(1), w[:-1]]), torch.cumsum(e3w, 0)


SPG_2D = ("un_b", "vn_b", "ub_b", "vb_b", "sshn", "hu_n", "hv_n", "r1_hu_n", "r1_hv_n", "ht_n", "rCdU_bot", "utau",
          "vtau", "emp", "rnf", "ub2_b", "vb2_b", "un_bf", "vn_bf")
SPG_OUT = ("ua_b", "va_b", "ssha", "un_adv", "vn_adv")


class Member:
    """One domain's fields in HBM and the calls of its time step."""

    def __init__(self, case, g, seed):
        h = self.h = nemo_hip.get()
        self.ctx, self.d = _grid(h, g)
        d, dt = self.d, _dt(case)
        self.sp, self.kind, self.kn = case["dtype"] == "f32", case["kind"], case["kn"]
        n2, n3 = d.jpi * d.jpj, d.jpi * d.jpj * d.jpk
        X = self.X = _inputs(case, g, d, seed)
        z = lambda n, t=dt: torch.zeros(n, dtype=t, device="cuda")  # noqa: E731
        if self.kind == "physics":
            X.update(pab=z(2 * n3), rn2b=z(n3), rhd=z(n3), rhdn=z(n3), rhop=z(n3), nmln=z(n2, torch.int32),
                     hmlp=z(n2, F64), hmlpt=z(n2, F64), uslp=z(n3), vslp=z(n3), wslpi=z(n3), wslpj=z(n3))
        elif self.kind == "adjoint":
            zu, zv, zw = z(n3), z(n3), z(n3)
            h.context_select(self.ctx)
            h.tra_adv_trp(X["un"], X["vn"], X["wn"], zu, zv, zw)
            self.model = autograd.TracerModel(h, zu, zv, zw, X["ahtu"], X["ahtv"], X["avt"], 2.0 * d.opts["rdt"],
                                              kn=(self.kn, self.kn), kt=KT)
        else:
            X.update({k: z(n2, F64) for k in SPG_OUT})
            if self.kind == "routines":
                X.update(zun=z(n3), zvn=z(n3), zwn=z(n3))
            else:
                X.update(ua=z(n3), va=z(n3), tsa=z(2 * n3), ah_wslp2=z(n3), akz=z(n3), hdivn=z(n3))
            self.spg = {k: X[k] for k in SPG_2D + SPG_OUT + ("ua", "va", "un", "vn")}

    def step(self, kt):
        h, X, sp = self.h, self.X, self.sp
        h.context_select(self.ctx)
        h.ssh_nxt(kt, X["un"], X["vn"], X["hdivn"], X["sshb"], X["emp_b"], X["emp"], X["ssha"], sp=sp)
        h.wzv(kt, X["hdivn"], X["wn"], sp=sp)
        h.step_dyn(kt, X["ub"], X["vb"], X["wn"], X["avm"], X["utau_b"], X["vtau_b"], self.spg, sp=sp)
        h.div_hor(kt, X["un"], X["vn"], X["hdivn"], sp=sp)
        h.wzv(kt, X["hdivn"], X["wn"], sp=sp)
        h.step_tra(kt, X["un"], X["vn"], X["wn"], X["tsb"], X["tsn"], X["tsa"], self.kn, self.kn, X["ahtu"], X["ahtv"],
                   X["uslp"], X["vslp"], X["wslpi"], X["wslpj"], X["ah_wslp2"], X["akz"], X["avt"], sp=sp)
        h.tra_nxt(kt, X["tsb"], X["tsn"], X["tsa"], sp=sp)
        h.dyn_nxt(kt, X["ub"], X["vb"], X["un"], X["vn"], X["ua"], X["va"], X["ua_b"], X["va_b"], X["un_adv"],
                  X["vn_adv"], X["ub_b"], X["vb_b"], X["un_b"], X["vn_b"], X["r1_hu_n"], X["r1_hv_n"], sp=sp)
        h.ssh_swp(kt, X["sshb"], X["sshn"], X["ssha"])

    def routines(self, kt):
        h, X, sp = self.h, self.X, self.sp
        h.context_select(self.ctx)
        h.dyn_adv(kt, X["un"], X["vn"], X["wn"], X["ua"], X["va"], sp=sp)
        h.dyn_vor(kt, X["un"], X["vn"], X["ua"], X["va"], sp=sp)
        h.dyn_spg_ts(kt, self.spg, sp=sp)
        h.dyn_zdf(kt, X["ub"], X["vb"], X["ua"], X["va"], X["avm"], X["rCdU_bot"], X["ua_b"], X["va_b"], X["utau"],
                  X["utau_b"], X["vtau"], X["vtau_b"], sp=sp)
        h.tra_adv_trp(X["un"], X["vn"], X["wn"], X["zun"], X["zvn"], X["zwn"], sp=sp)
        h.tra_adv_fct(kt, 1, "TRA", 2.0 * self.d.opts["rdt"], X["zun"], X["zvn"], X["zwn"], X["tsb"], X["tsn"], X["tsa"],
                      2, self.kn, self.kn, sp=sp)
        h.tra_ldf_lap(kt, 1, "TRA", X["ahtu"], X["ahtv"], X["tsb"], X["tsa"], 2, 1, sp=sp)
        h.tra_zdf(kt, X["tsb"], X["tsa"], X["avt"], X["avt"], sp=sp)

    def physics(self, kt):
        h, X, sp = self.h, self.X, self.sp
        h.context_select(self.ctx)
        h.rab_3d(X["tsb"], X["pab"], X["gdept"], sp=sp)
        h.bn2(X["tsb"], X["pab"], X["rn2b"], X["gdept"], X["gdepw"], sp=sp)
        h.zdf_mxl(kt, X["rn2b"], X["gdept"], X["gdepw"], configs.nlb10(self.d), X["nmln"], X["hmlp"], X["hmlpt"],
                  rho_c=RHO_C, sp=sp)
        h.eos_insitu(X["tsb"], X["rhd"], X["gdept"], sp=sp)
        h.ldf_slp(kt, X["rhd"], X["rn2b"], X["gdept"], X["gdepw"], X["nmln"], X["hmlp"], X["hmlpt"], RN_SLPMAX,
                  X["uslp"], X["vslp"], X["wslpi"], X["wslpj"], sp=sp)
        h.eos_insitu_pot(X["tsn"], X["rhdn"], X["rhop"], X["gdept"], sp=sp)
        h.dyn_ldf_lap(kt, X["ub"], X["vb"], X["ua"], X["va"], 1, X["ahmt"], X["ahmf"], sp=sp)
        h.hpg_zco(kt, X["rhdn"], X["ua"], X["va"], sp=sp)


class State:
    def __init__(self, case, seed):
        self.kind, self.kt = case["kind"], KT
        self.members = [Member(case, g, int(seed) * 64 + q) for q, g in enumerate(_members(case))]
        self.plan = None
        if self.kind == "ensemble":
            h = self.members[0].h
            h.plan_begin()
            for m in self.members:
                m.step(KT)
            self.plan = h.plan_end()

    def __del__(self):
        if getattr(self, "plan", None) is not None:
            self.members[0].h.plan_free(self.plan)


def prepare(case, seed):
    return State(case, seed)


STEP_OUT = ("tsn", "tsb", "un", "vn", "ub", "vb", "wn", "sshn", "sshb", "un_b", "vn_b", "ub_b", "vb_b")
ROUTINES_OUT = ("ua", "va", "un", "vn", "tsa", "zwn", "ssha", "ua_b", "va_b", "un_adv", "vn_adv", "un_bf")
PHYSICS_OUT = ("pab", "rn2b", "nmln", "hmlp", "hmlpt", "rhd", "uslp", "vslp", "wslpi", "wslpj", "rhdn", "rhop", "ua",
               "va")


def _out_names(case):
    if case["kind"] == "ensemble":
        return ("tsn", "un", "vn", "ub", "wn", "sshn", "un_b")
    return {"step": STEP_OUT, "routines": ROUTINES_OUT, "physics": PHYSICS_OUT}[case["kind"]]


def run(state):
    s, m = state, state.members[0]
    if s.kind == "ensemble":
        m.h.plan_launch(s.plan)
        return [{k: q.X[k] for k in _out_names({"kind": s.kind})} for q in s.members]
    if s.kind == "adjoint":
        m.h.context_select(m.ctx)
        tb, tn = (m.X[k].detach().requires_grad_() for k in ("tsb", "tsn"))
        nb, nn = autograd.TracerStep.apply(tb, tn, m.model)
        gb, gn = torch.autograd.grad((nb, nn), (tb, tn), (m.X["gb"], m.X["gn"]))
        return {"tb": nb.detach(), "tn": nn.detach(), "grad_tb": gb, "grad_tn": gn}
    getattr(m, s.kind)(s.kt)
    s.kt += 1
    return {k: m.X[k] for k in _out_names({"kind": s.kind})}


# 3D arrays a pass reads and writes once each, and operations per cell (both tracers); 2D arrays of FP64
WORK = {"step": (28, 900, 40), "ensemble": (28, 900, 40), "routines": (26, 700, 40), "physics": (24, 600, 6),
        "adjoint": (14, 600, 0)}


def work(case):
    arrays, flops, flat = WORK[case["kind"]]
    size = 8 if case["dtype"] == "f64" else 4
    n3 = sum(g["jpi"] * g["jpj"] * g["jpk"] for g in _members(case))
    n2 = n3 // case["jpk"]
    sub = 44 * 120 if case["kind"] in ("step", "ensemble", "routines") else 0   # the barotropic sub-steps
    return {"bytes": arrays * n3 * size + flat * n2 * 8, "flops": flops * n3 + sub * n2}


# about four times the largest error against exact() over the listed and some drawn cases: FP64 4e-14 (w, a sum of
# cancelling terms); FP32 storage 2.3e-5 in w, 2.9e-6 in the slopes, 1e-7 elsewhere
def tolerance(case):
    if case["dtype"] == "f64":
        return {"rel": 2e-13, "max": 1e-10}
    return {"rel": {"step": 1e-4, "ensemble": 1e-4, "routines": 1e-6, "physics": 1.2e-5}[case["kind"]]}


# ----------------------------------------------------------------------------
# the same passes in plain torch, FP64.  Arrays are (..., k, j, i); xp(a) holds
# a(i+1) at i (the last point wraps and is never used), xm, yp, ym alike.
# ----------------------------------------------------------------------------
def xp(a):
    return a.roll(-1, -1)


def xm(a):
    return a.roll(1, -1)


def yp(a):
    return a.roll(-1, -2)


def ym(a):
    return a.roll(1, -2)


def kdown(a):
    """a(k+1) at level k, zero at the last level"""
    return torch.cat([a[..., 1:, :, :], torch.zeros_like(a[..., :1, :, :])], -3)


def kup(a):
    """a(k-1) at level k, a(1) at the first"""
    return torch.cat([a[..., :1, :, :], a[..., :-1, :, :]], -3)


def lbc(a, jperio, nat):
    """the serial lateral boundary fill: cyclic copies, or zero on a closed side (F-points keep their first row)"""
    a = a.clone()
    if jperio in (1, 7):
        a[..., 0], a[..., -1] = a[..., -2].clone(), a[..., 1].clone()
    else:
        if nat != "F":
            a[..., 0] = 0
        a[..., -1] = 0
    if jperio in (2, 7):
        a[..., 0, :], a[..., -1, :] = a[..., -2, :].clone(), a[..., 1, :].clone()
    else:
        if nat != "F":
            a[..., 0, :] = 0
        a[..., -1, :] = 0
    return a


class Masks:
    def __init__(self, d, device):
        T2 = lambda n: torch.from_numpy(d.arrays[n].T.copy()).to(device)  # noqa: E731
        kt, kb = T2("k_top").long(), T2("k_bot").long()
        k = torch.arange(1, d.jpk + 1, device=device)[:, None, None]
        t = lbc(((kt != 0) & (k >= kt) & (k <= kb)).to(F64), d.jperio, "T")
        cut = torch.zeros(d.jpj, d.jpi, device=device, dtype=F64)
        cut[:-1, :-1] = 1
        self.t, self.u, self.v = t, lbc(t * xp(t) * cut, d.jperio, "U"), lbc(t * yp(t) * cut, d.jperio, "V")
        self.f = lbc(t * xp(t) * yp(t) * xp(yp(t)) * cut, d.jperio, "F")
        self.w, self.wu, self.wv = (a * kup(a) for a in (t, self.u, self.v))
        self.mikt, self.mbkt = kt.clamp(min=1), kb.clamp(min=1)
        lb = lambda a, nat: lbc(a.to(F64), d.jperio, nat).round().long().clamp(min=1)  # noqa: E731
        c = cut.long()
        self.mbku = lb(torch.minimum(xp(self.mbkt), self.mbkt) * c, "U")
        self.mbkv = lb(torch.minimum(yp(self.mbkt), self.mbkt) * c, "V")
        self.ss, self.ssu, self.ssv = (a.amax(0) for a in (self.t, self.u, self.v))
        self.inner = torch.zeros_like(cut)
        self.inner[1:-1, 1:-1] = 1


class Exact:
    """One domain's operators; X holds its fields as FP64 (k, j, i) tensors."""

    def __init__(self, case, d, X, device="cuda"):
        self.d, self.case, self.jperio, self.o = d, case, d.jperio, d.opts
        self.m = Masks(d, device)
        self.e = {n: torch.from_numpy(d.arrays[n].T.copy()).to(device) for n in abi.DOMAIN_2D_FIELDS
                  if d.arrays.get(n) is not None}
        self.e3t, self.e3w = (torch.from_numpy(a).to(device)[:, None, None] for a in (d.e3t_1d, d.e3w_1d))
        s2, s3 = (d.jpj, d.jpi), (d.jpk, d.jpj, d.jpi)
        sizes = {d.jpi * d.jpj: s2, d.jpk * d.jpi * d.jpj: s3, 2 * d.jpk * d.jpi * d.jpj: (2,) + s3}
        self.X = {k: v.double().reshape(sizes[v.numel()]).clone() for k, v in X.items()}
        self.z2, self.z3 = torch.zeros(s2, dtype=F64, device=device), torch.zeros(s3, dtype=F64, device=device)
        self.p2dt = 2.0 * self.o["rdt"]
        self.km = torch.ones(d.jpk, 1, 1, dtype=F64, device=device)    # levels 1..jpkm1
        self.km[-1] = 0

    def lbc(self, a, nat):
        return lbc(a, self.jperio, nat)

    def at(self, a, k):
        """a at each column's level k (1-based)"""
        return a.gather(0, (k - 1)[None])[0]

    # momentum ---------------------------------------------------------------
    def dyn_adv(self, un, vn, wn, ua, va):
        e, m = self.e, self.m
        ke = 0.25 * (un ** 2 + xm(un) ** 2 + vn ** 2 + ym(vn) ** 2)
        zww = 0.25 * e["e1e2t"] * wn * self.km
        zww[0] = 0
        wu, wv = (xp(zww) + zww) * (kup(un) - un), (yp(zww) + zww) * (kup(vn) - vn)
        du = -(xp(ke) - ke) / e["e1u"] - (wu + kdown(wu)) * e["r1_e1e2u"] / self.e3t
        dv = -(yp(ke) - ke) / e["e2v"] - (wv + kdown(wv)) * e["r1_e1e2v"] / self.e3t
        on = m.inner * self.km
        return ua + du * on, va + dv * on

    def dyn_vor(self, un, vn, ua, va):
        e, m = self.e, self.m
        curl = e["ff_f"] + (xp(e["e2v"] * vn) - e["e2v"] * vn - yp(e["e1u"] * un) + e["e1u"] * un) * e["r1_e1e2f"]
        on = m.inner * self.km
        if self.case["vor"] == "ene":
            y, x = e["e1v"] * vn, e["e2u"] * un
            y, x = y + xp(y), x + yp(x)
            return (ua + on * 0.25 * e["r1_e1u"] * (ym(curl) * ym(y) + curl * y),
                    va - on * 0.25 * e["r1_e2v"] * (xm(curl) * xm(x) + curl * x))
        n = yp(m.t) + xp(yp(m.t)) + m.t + xp(m.t)
        f = self.lbc(curl * torch.where(n > 0, n / (self.e3t * n).clamp(min=1e-300), 0.0), "F")
        return self._triads(f, e["e2u"] * self.e3t * un, e["e1v"] * self.e3t * vn, ua, va, on)

    def _triads(self, f, x, y, ua, va, on):
        e = self.e
        ne, nw = xm(f) + f + ym(f), xm(ym(f)) + xm(f) + f
        se, sw = f + ym(f) + xm(ym(f)), ym(f) + xm(ym(f)) + xm(f)
        du = e["r1_e1u"] / 12 * (ne * y + xp(nw) * xp(y) + se * ym(y) + xp(sw) * xp(ym(y)))
        dv = -e["r1_e2v"] / 12 * (yp(sw) * xm(yp(x)) + yp(se) * yp(x) + nw * xm(x) + ne * x)
        return ua + du * on, va + dv * on

    def dyn_spg_ts(self, ua, va, un, vn, X):
        """phases 1 to 3; returns ua, va, un, vn and updates the 2D fields of X"""
        e, m, o, in_ = self.e, self.m, self.o, self.m.inner
        rau0, jp = o["rau0"], self.jperio
        een = self.case["vor"] == "een"
        ht, hu, hv, r1u, r1v = (X[k] for k in ("ht_n", "hu_n", "hv_n", "r1_hu_n", "r1_hv_n"))
        cut = torch.zeros_like(in_)
        cut[:-1, :-1] = 1
        if een:
            s, n = ht + xp(ht) + yp(ht) + xp(yp(ht)), m.ss + xp(m.ss) + yp(m.ss) + xp(yp(m.ss))
            z = s / n.clamp(min=1.0)
            f = lbc(torch.where(z != 0, e["ff_f"] / torch.where(z != 0, z, 1.0), 0.0) * cut, jp, "F")
        else:
            z = lbc((self.e3t * m.u * yp(m.u) * self.km).sum(0) * torch.cat([torch.ones_like(in_[:-1]), in_[-1:] * 0]),
                    jp, "F")
            f = torch.where(z != 0, e["ff_f"] / torch.where(z != 0, z, 1.0), 0.0)

        def coriolis(x, y):
            if een:
                return self._triads(f, x, y, 0.0, 0.0, 1.0)
            yy, xx = y + xp(y), x + yp(x)
            return (0.25 * e["r1_e1u"] * (ym(f) * ym(yy) + f * yy),
                    -0.25 * e["r1_e2v"] * (xm(f) * xm(xx) + f * xx))
        fu = (self.e3t * ua * m.u * self.km).sum(0) * r1u
        fv = (self.e3t * va * m.v * self.km).sum(0) * r1v
        ua, va = ua - fu * m.u * in_ * self.km, va - fv * m.v * in_ * self.km
        cu, cv = coriolis(X["un_b"] * hu * e["e2u"], X["vn_b"] * hv * e["e1v"])
        dru, drv = 0.5 * (xp(X["rCdU_bot"]) + X["rCdU_bot"]), 0.5 * (yp(X["rCdU_bot"]) + X["rCdU_bot"])
        fu = fu - cu * m.ssu + r1u * dru * (self.at(un, m.mbku) - X["un_b"]) + X["utau"] * r1u / rau0
        fv = fv - cv * m.ssv + r1v * drv * (self.at(vn, m.mbkv) - X["vn_b"]) + X["vtau"] * r1v / rau0
        fs = (X["emp"] - X["rnf"]) / rau0
        w1, w2 = _bt_weights(o["nn_baro"])
        dt = o["rdt"] / o["nn_baro"]
        u, v, h = [X["un_b"]] + 2 * [self.z2], [X["vn_b"]] + 2 * [self.z2], [X["sshn"]] + 2 * [self.z2]
        ssha, ua_b, va_b, un_adv, vn_adv = (self.z2.clone() for _ in range(5))
        for n in range(len(w1)):
            a = (1.0, 0.0, 0.0) if n < 2 else (1.781105, -1.06221, 0.281105)
            x = e["e2u"] * sum(c * q for c, q in zip(a, u)) * hu
            y = e["e1v"] * sum(c * q for c, q in zip(a, v)) * hv
            un_adv += w2[n] * x * e["r1_e2u"]
            vn_adv += w2[n] * y * e["r1_e1v"]
            ha = lbc((h[0] - dt * (fs + (x - xm(x) + y - ym(y)) * e["r1_e1e2t"])) * m.ss, jp, "T")
            ssha += w1[n] * ha
            b = ((1.0, 0.0, 0.0, 0.0) if n == 0 else (1.0833333333333, -0.1666666666666, 0.0833333333333, 0.0)
                 if n == 1 else (0.614, 0.285, 0.088, 0.013))
            p = b[0] * ha + b[1] * h[0] + b[2] * h[1] + b[3] * h[2]
            cu, cv = coriolis(x, y)
            gu, gv = -o["grav"] * (xp(p) - p) * e["r1_e1u"], -o["grav"] * (yp(p) - p) * e["r1_e2v"]
            nu = lbc((u[0] + dt * (gu + cu + dru * u[0] * r1u + fu)) * m.ssu, jp, "U")
            nv = lbc((v[0] + dt * (gv + cv + drv * v[0] * r1v + fv)) * m.ssv, jp, "V")
            ua_b += w1[n] * nu
            va_b += w1[n] * nv
            u, v, h = [nu] + u[:2], [nv] + v[:2], [ha] + h[:2]
        at = o["rn_atfp"]
        for adv, b2, bf in ((un_adv, "ub2_b", "un_bf"), (vn_adv, "vb2_b", "vn_bf")):
            raw = adv.clone()
            adv.copy_(0.5 * (X[b2] + raw - at * X[bf]))
            X[bf], X[b2] = at * X[bf] + (raw - X[b2]), raw
        X.update(ssha=ssha, ua_b=ua_b, va_b=va_b, un_adv=un_adv, vn_adv=vn_adv)
        ua = ua + (ua_b - X["ub_b"]) / self.p2dt * self.km
        va = va + (va_b - X["vb_b"]) / self.p2dt * self.km
        un = torch.where(self.km > 0, (un + un_adv * r1u - X["un_b"]) * m.u, un)
        vn = torch.where(self.km > 0, (vn + vn_adv * r1v - X["vn_b"]) * m.v, vn)
        return ua, va, un, vn

    def dyn_zdf(self, pb, pa, avm, c, X):
        """one velocity component: c = "u" or "v" """
        m, o, r = self.m, self.o, self.p2dt
        msk, wm, ikb = (m.u, m.wu, m.mbku) if c == "u" else (m.v, m.wv, m.mbkv)
        nb = xp if c == "u" else yp
        ab, tau = X[c + "a_b"], 0.5 * (X[c + "tau_b"] + X[c + "tau"])
        a = ((pb + r * pa) * msk - ab) * msk * self.km + pa * (1 - self.km)
        e3 = self.e3t[:, 0, 0]
        cs = 0.5 * (nb(X["rCdU_bot"]) + X["rCdU_bot"])
        n = self.d.jpk - 1
        kk = torch.arange(1, self.d.jpk + 1, device=a.device)[:, None, None]
        bot = (kk == ikb).to(F64) * cs * r / self.e3t
        b = a + bot * ab
        b[0] = b[0] + r * tau / (e3[0] * o["rau0"]) * msk[0]
        av = -0.5 * r * (nb(avm) + avm) / self.e3w * wm
        lo, up = av / self.e3t, kdown(av) / self.e3t
        lo[0] = 0
        x = _thomas(lo[:n], 1 - lo[:n] - up[:n] - bot[:n], up[:n], b[:n])
        return torch.where(m.inner * self.km > 0, torch.cat([x, a[n:]]), a)

    # tracers ------------------------------------------------------------------
    def transports(self, un, vn, wn):
        e = self.e
        return e["e2u"] * self.e3t * un * self.km, e["e1v"] * self.e3t * vn * self.km, e["e1e2t"] * wn * self.km

    def fct(self, u, v, w, tb, tn, kn, p2dt, frozen=None, keep=None):
        """the trend of one tracer; frozen: the limiter's factors, keep: a list that receives them"""
        e, m, jp = self.e, self.m, self.jperio
        r1, e3, on = e["r1_e1e2t"], self.e3t, m.inner * self.km
        pos, neg = lambda a: 0.5 * (a + a.abs()), lambda a: 0.5 * (a - a.abs())  # noqa: E731
        hu, hv = pos(u) * tb + neg(u) * xp(tb), pos(v) * tb + neg(v) * yp(tb)
        hw = (pos(w) * tb + neg(w) * kup(tb)) * m.w * self.km
        hw = torch.cat([(w[:1] * tb[:1]), hw[1:]])
        low = -(hu - xm(hu) + hv - ym(hv) + hw - kdown(hw)) * r1
        trend = low / e3 * m.t * on
        zwi = lbc((e3 * tb + p2dt * low) / e3 * m.t * on, jp, "T")
        fu, fv = tn + xp(tn), tn + yp(tn)
        if kn == 4:
            a, b = (xp(tn) - tn) * m.u, (yp(tn) - tn) * m.v
            a, b = lbc((a + xm(a)) / 6, jp, "T"), lbc((b + ym(b)) / 6, jp, "T")
            fu, fv = fu + a - xp(a), fv + b - yp(b)
            fw = self._compact(tn)
        else:
            fw = 0.5 * (tn + kup(tn))
        ax, ay = lbc(0.5 * u * fu - hu, jp, "U"), lbc(0.5 * v * fv - hv, jp, "V")
        az = (w * fw - hw) * m.w * on
        az = torch.cat([torch.zeros_like(az[:1]), az[1:]])
        if frozen is None:
            frozen = self._zalesak(tb, zwi, ax, ay, lbc(az, jp, "T"), p2dt)
            if keep is not None:
                keep.extend(frozen)
        cx, cy, cz = frozen
        ax, ay, az = lbc(ax * cx, jp, "U"), lbc(ay * cy, jp, "V"), az * cz
        return trend - (ax - xm(ax) + ay - ym(ay) + az - kdown(az)) * r1 / e3 * on

    def _compact(self, tn):
        """the compact vertical interpolation to w-levels"""
        n, ikb = self.d.jpk - 1, self.m.mbkt
        k = torch.arange(2, n + 1, device=tn.device)[:, None, None]
        end = (k == 2) | (k == ikb)
        wm = self.m.w[1:n]
        mean = tn[1:n] + tn[: n - 1]
        off = torch.where(end, 0.0, wm)
        x = _thomas(off, torch.where(end, 1.0, 3 * wm + 1), off, torch.where(end, 0.5 * mean, 3 * wm * mean))
        return torch.cat([tn[:1] * 0, x, tn[:1] * 0])

    def _zalesak(self, before, after, ax, ay, az, p2dt):
        m, jp, on = self.m, self.jperio, self.m.inner * self.km
        wet = m.t > 0
        big = 1e40
        up = torch.where(wet, torch.maximum(before, after), -big)
        do = torch.where(wet, torch.minimum(before, after), big)
        dn = lambda a: torch.cat([a[1:], a[-1:]])  # noqa: E731
        ext = lambda a, f: f(f(f(a, xm(a)), f(xp(a), ym(a))), f(f(yp(a), kup(a)), dn(a)))  # noqa: E731
        pos, neg = lambda a: a.clamp(min=0), lambda a: a.clamp(max=0)  # noqa: E731
        zp = pos(xm(ax)) - neg(ax) + pos(ym(ay)) - neg(ay) + pos(kdown(az)) - neg(az)
        zn = pos(ax) - neg(xm(ax)) + pos(ay) - neg(ym(ay)) + pos(az) - neg(kdown(az))
        vol = self.e["e1e2t"] * self.e3t / p2dt
        bu = lbc((ext(up, torch.maximum) - after) / (zp + 1e-15) * vol * on, jp, "T")
        bd = lbc((after - ext(do, torch.minimum)) / (zn + 1e-15) * vol * on, jp, "T")
        one = torch.ones_like(bu)
        fac = lambda a, nb: torch.where(a >= 0, torch.minimum(one, torch.minimum(bd, nb(bu))),  # noqa: E731
                                        torch.minimum(one, torch.minimum(bu, nb(bd))))
        return fac(ax, xp), fac(ay, yp), fac(az, kup)

    def ldf_lap(self, tb, ahu, ahv):
        e, on = self.e, self.m.inner * self.km
        fu, fv = ahu * e["e2_e1u"] * self.e3t * (xp(tb) - tb), ahv * e["e1_e2v"] * self.e3t * (yp(tb) - tb)
        return (fu - xm(fu) + fv - ym(fv)) / (e["e1e2t"] * self.e3t) * on

    def iso_coef(self, ahu, ahv, wslpi, wslpj):
        m = self.m
        mu = m.w / (kup(m.u) + xm(m.u) + xm(kup(m.u)) + m.u).clamp(min=1)
        mv = m.w / (kup(m.v) + ym(m.v) + ym(kup(m.v)) + m.v).clamp(min=1)
        hu = (kup(ahu) + xm(ahu) + xm(kup(ahu)) + ahu) * mu
        hv = (kup(ahv) + ym(ahv) + ym(kup(ahv)) + ahv) * mv
        a = (hu * wslpi ** 2 + hv * wslpj ** 2) * m.inner * self.km
        a[0] = 0
        return a

    def ldf_iso(self, tb, ahu, ahv, us, vs, wsi, wsj, ah, akz):
        e, m, on = self.e, self.m, self.m.inner * self.km
        low = torch.ones_like(self.km)                 # w-levels 2..jpkm1
        low[0] = low[-1] = 0
        dk = (kup(tb) - tb) * m.w                      # at w-level k
        dk[0] = 0
        w0, w1 = m.w, kdown(m.w)
        d1 = kdown(dk)
        d0 = torch.cat([d1[:1], dk[1:]])               # zdkt(1) = zdk1t(1)

        def face(nb, ah_, s, ratio, width, msk):
            n = 1 / (nb(w0) + w1 + nb(w1) + w0).clamp(min=1)
            return (ah_ * ratio * self.e3t * (nb(tb) - tb) * msk
                    - ah_ * width * s * n * (nb(d0) + d1 + nb(d1) + d0)) * msk
        fu = face(xp, ahu, us, e["e2_e1u"], e["e2u"], m.u)
        fv = face(yp, ahv, vs, e["e1_e2v"], e["e1v"], m.v)
        gi, gj = (xp(tb) - tb) * m.u, (yp(tb) - tb) * m.v

        def wpart(g, back, msk, ah_, s, width):
            n = m.w / (kup(msk) + back(msk) + back(kup(msk)) + msk).clamp(min=1)
            hw = (kup(ah_) + back(ah_) + back(kup(ah_)) + ah_) * n
            return -hw * width * n * s * (kup(g) + back(g) + back(kup(g)) + g)
        fw = (wpart(gi, xm, m.u, ahu, wsi, e["e2t"]) + wpart(gj, ym, m.v, ahv, wsj, e["e1t"])
              + e["e1e2t"] / self.e3w * m.w * (ah - akz) * (kup(tb) - tb)) * low
        return (fu - xm(fu) + fv - ym(fv) + fw - kdown(fw)) * e["r1_e1e2t"] / self.e3t * on

    def tra_zdf(self, tb, ta, kz, p2dt):
        """the after tracer of the interior"""
        n, m = self.d.jpk - 1, self.m
        kz = kz.clone()
        kz[0] = 0
        lo, up = -p2dt * kz[:n] / self.e3w[:n], -p2dt * kz[1:] / self.e3w[1:]
        rhs = (self.e3t * (tb + p2dt * ta))[:n]
        x = _thomas(lo, self.e3t[:n] - lo - up, up, rhs, m.t[:n])
        return torch.where(m.inner * self.km > 0, torch.cat([x, ta[n:]]), ta)

    # time-step closure ----------------------------------------------------------
    def div_hor(self, un, vn):
        e = self.e
        x, y = e["e2u"] * self.e3t * un, e["e1v"] * self.e3t * vn
        return self.lbc((x - xm(x) + y - ym(y)) * e["r1_e1e2t"] / self.e3t * self.km, "T")

    def wzv(self, hdiv):
        return -((self.e3t * hdiv * self.m.t * self.km).flip(0).cumsum(0)).flip(0)

    # passes -----------------------------------------------------------------------
    def step(self):
        X, m, o = self.X, self.m, self.o
        at = o["rn_atfp"]
        un, vn = X["un"], X["vn"]
        wn = self.wzv(self.div_hor(un, vn))
        ua, va = self.dyn_adv(un, vn, wn, self.z3, self.z3)
        ua, va = self.dyn_vor(un, vn, ua, va)
        ua, va, un, vn = self.dyn_spg_ts(ua, va, un, vn, X)
        wn = self.wzv(self.div_hor(un, vn))
        ua, va = self.dyn_zdf(X["ub"], ua, X["avm"], "u", X), self.dyn_zdf(X["vb"], va, X["avm"], "v", X)
        tr = self.transports(un, vn, wn)
        ah = self.iso_coef(X["ahtu"], X["ahtv"], X["wslpi"], X["wslpj"])
        tsa = []
        for q in range(2):
            tb, tn = X["tsb"][q], X["tsn"][q]
            ta = self.fct(*tr, tb, tn, self.case["kn"], self.p2dt)
            ta = ta + self.ldf_iso(tb, X["ahtu"], X["ahtv"], X["uslp"], X["vslp"], X["wslpi"], X["wslpj"], ah, ah)
            ta = self.tra_zdf(tb, ta, X["avt"] + ah * self.km, self.p2dt)
            tsa.append(torch.where(ta < 0, 0.1, ta) if q == 1 else ta)
        ta, tb, tn = torch.stack(tsa), X["tsb"], X["tsn"]
        on = m.inner * self.km
        nb = torch.where(on > 0, tn + at * (ta - 2 * tn + tb), tb)
        nn = torch.where(on > 0, ta, tn)
        out = dict(tsb=self.lbc(nb, "T"), tsn=self.lbc(nn, "T"), wn=wn)
        for c, a, b, n, lb in (("u", ua, X["ub"], un, "U"), ("v", va, X["vb"], vn, "V")):
            msk, r1 = (m.u, X["r1_hu_n"]) if c == "u" else (m.v, X["r1_hv_n"])
            s = lambda q: (self.e3t * q * msk * self.km).sum(0) * r1  # noqa: E731
            a = torch.where(on > 0, (a - s(a) + X[c + "a_b"]) * msk, a)
            a = self.lbc(a, lb)
            f = torch.where(self.km > 0, n + at * (b - 2 * n + a), b)
            f = torch.where(self.km > 0, f - (s(f) - X[c + "n_b"]) * msk, f)
            n = torch.where(self.km > 0, a, n)
            out.update({c + "n": n, c + "b": f, c + "n_b": s(n), c + "b_b": s(f)})
        out["sshb"] = X["sshn"] + at * (X["sshb"] - 2 * X["sshn"] + X["ssha"])
        out["sshn"] = X["ssha"]
        return out

    def routines(self):
        X = self.X
        ua, va = self.dyn_adv(X["un"], X["vn"], X["wn"], X["ua"], X["va"])
        ua, va = self.dyn_vor(X["un"], X["vn"], ua, va)
        ua, va, un, vn = self.dyn_spg_ts(ua, va, X["un"], X["vn"], X)
        ua, va = self.dyn_zdf(X["ub"], ua, X["avm"], "u", X), self.dyn_zdf(X["vb"], va, X["avm"], "v", X)
        tr = self.transports(un, vn, X["wn"])
        tsa = []
        for q in range(2):
            tb = X["tsb"][q]
            ta = X["tsa"][q] + self.fct(*tr, tb, X["tsn"][q], self.case["kn"], self.p2dt)
            ta = self.tra_zdf(tb, ta + self.ldf_lap(tb, X["ahtu"], X["ahtv"]), X["avt"], self.p2dt)
            tsa.append(torch.where(ta < 0, 0.1, ta) if q == 1 else ta)
        out = {k: X[k] for k in ("ssha", "ua_b", "va_b", "un_adv", "vn_adv", "un_bf")}
        out.update(ua=ua, va=va, un=un, vn=vn, tsa=torch.stack(tsa), zwn=tr[2])
        return out

    def adjoint(self):
        X, at, p2dt = self.X, self.o["rn_atfp"], self.p2dt
        tr = self.transports(X["un"], X["vn"], X["wn"])
        tb, tn = X["tsb"].requires_grad_(), X["tsn"].requires_grad_()
        fac = []
        with torch.no_grad():
            self.fct(*tr, tb, tn, self.case["kn"], p2dt, keep=fac)
        ta = self.fct(*tr, tb, tn, self.case["kn"], p2dt, frozen=fac) + self.ldf_lap(tb, X["ahtu"], X["ahtv"])
        ta = self.tra_zdf(tb, ta, X["avt"], p2dt)
        on = self.m.inner * self.km
        nb = self.lbc(torch.where(on > 0, tn + at * (ta - 2 * tn + tb), tb), "T")
        nn = self.lbc(torch.where(on > 0, ta, tn), "T")
        gb, gn = torch.autograd.grad((nb, nn), (tb, tn), (X["gb"], X["gn"]))
        return {"tb": nb.detach(), "tn": nn.detach(), "grad_tb": gb, "grad_tn": gn}

    def density(self, ts, dep):
        """density anomaly from rau0, kg/m3, its value at the surface pressure, and rau0 (alpha, beta)"""
        rau0 = self.o["rau0"]
        if self.case["eos"] == "seos":
            c = abi.SEOS_DEFAULTS
            a0, b0, l1, l2, m1, m2, nu = (c[k] for k in abi.EOS_REAL_FIELDS)
            t, s = ts[0] - 10.0, ts[1] - 35.0
            pot = -a0 * (1 + 0.5 * l1 * t) * t + b0 * (1 - 0.5 * l2 * s) * s - nu * t * s
            return (pot - (a0 * m1 * t + b0 * m2 * s) * dep, pot + rau0,
                    a0 * (1 + l1 * t + m1 * dep) + nu * s, b0 * (1 - l2 * s - m2 * dep) - nu * t)
        t, z = ts[0] / 40.0, dep * 1e-4
        s = torch.sqrt((ts[1] + 32.0).abs() * (0.875 / 35.16504))
        pot = rho = rt = rs = torch.zeros_like(t)
        for k, table in enumerate(TEOS10):
            for j, row in enumerate(table):
                for i, c in enumerate(row):
                    mono = c * z ** k
                    rho = rho + mono * t ** j * s ** i
                    if k == 0:
                        pot = pot + mono * t ** j * s ** i
                    if j:
                        rt = rt - mono * j * t ** (j - 1) * s ** i / 40.0
                    if i:
                        rs = rs + mono * t ** j * i * s ** (i - 2) * (0.5 * 0.875 / 35.16504)
        return rho - rau0, pot, rt, rs

    def physics(self):
        X, m, o, e = self.X, self.m, self.o, self.e
        rau0, on, g = o["rau0"], m.inner * self.km, o["grav"]
        dep, depw = X["gdept"], X["gdepw"]
        rd, _, al, be = self.density(X["tsb"], dep)
        km = m.t * self.km
        out = {"pab": torch.stack([al, be]) / rau0 * km, "rhd": rd / rau0 * km}
        al, be = out["pab"]
        # N2 at w-levels 2..jpkm1
        r = (depw - dep) / torch.where(kup(dep) != dep, kup(dep) - dep, 1.0)
        aw, bw = al * (1 - r) + kup(al) * r, be * (1 - r) + kup(be) * r
        T, S = X["tsb"]
        n2 = g * (aw * (kup(T) - T) - bw * (kup(S) - S)) / self.e3w * m.w * self.km
        n2[0] = 0
        out["rn2b"] = n2
        # mixed layer
        nl = configs.nlb10(self.d)
        nm, hint = torch.full_like(m.mbkt, nl), self.z2
        for k in range(nl, self.d.jpk):
            hint = hint + n2[k - 1].clamp(min=0) * self.e3w[k - 1]
            nm = torch.where(hint < g * RHO_C / rau0, m.mbkt.clamp(max=k) + 1, nm)
        out.update(nmln=None, hmlp=self.at(depw, nm) * m.ss, hmlpt=self.at(dep, nm - 1) * m.ss)
        self._slopes(out, out["rhd"], n2, dep, depw, nm)
        rd, pot, _, _ = self.density(X["tsn"], dep)
        out["rhdn"], out["rhop"] = rd / rau0 * km, pot * km
        # viscosity
        ub, vb = X["ub"], X["vb"]
        cur = X["ahmf"] * self.e3t * e["r1_e1e2f"] * (xp(e["e2v"] * vb) - e["e2v"] * vb - yp(e["e1u"] * ub) + e["e1u"] * ub)
        x, y = e["e2u"] * self.e3t * ub, e["e1v"] * self.e3t * vb
        div = X["ahmt"] * e["r1_e1e2t"] / self.e3t * (x - xm(x) + y - ym(y))
        ua = X["ua"] + on * (-(cur - ym(cur)) * e["r1_e2u"] / self.e3t + (xp(div) - div) * e["r1_e1u"])
        va = X["va"] + on * ((cur - xm(cur)) * e["r1_e1v"] / self.e3t + (yp(div) - div) * e["r1_e2v"])
        # pressure gradient
        rh = out["rhdn"]
        s = rh + kup(rh)
        s = torch.cat([rh[:1], s[1:]])
        c = -0.5 * g * self.e3w
        out["ua"] = ua + on * torch.cumsum(c * (xp(s) - s), 0) * e["r1_e1u"]
        out["va"] = va + on * torch.cumsum(c * (yp(s) - s), 0) * e["r1_e2v"]
        return out

    def _slopes(self, out, prd, n2, dep, depw, nm):
        m, e, jp, g = self.m, self.e, self.jperio, self.o["grav"]
        eps, jpkm1 = 1e-20, self.d.jpk - 1
        gu, gv = m.u * (xp(prd) - prd), m.v * (yp(prd) - prd)
        dz = -1 / g * (prd + 1) * (n2 + kdown(n2)) * (1 - 0.5 * kdown(m.t))
        dz[0] = 0
        kk = torch.arange(1, self.d.jpk + 1, device=prd.device)[:, None, None]
        oml = (kk <= nm - 1).to(F64)
        lim = lambda b, a, h, c: torch.minimum(torch.minimum(b, -c * a.abs()), -7e3 / h * a.abs())  # noqa: E731

        def filt(a):
            return (xm(ym(a)) + xp(ym(a)) + xm(yp(a)) + xp(yp(a)) + 2 * (ym(a) + xm(a) + xp(a) + yp(a)) + 4 * a) / 16
        lev = torch.ones_like(self.km)                 # levels 2..jpkm1
        lev[0] = lev[-1] = 0
        for name, nb, grad, r1e, msk, nat, across in (("uslp", xp, gu, e["r1_e1u"], m.u, "U", (ym, yp)),
                                                      ("vslp", yp, gv, e["r1_e2v"], m.v, "V", (xm, xp))):
            za = grad * r1e
            slope = lambda a, b, h, mk: a / (lim(b, a, h, 1 / RN_SLPMAX) - eps) * mk  # noqa: E731
            zb = 0.5 * (dz + nb(dz))
            ik = torch.maximum(nm, nb(nm)).clamp(1, jpkm1)
            ml = slope(self.at(za, ik), self.at(zb, ik), self.e3t[:, 0, 0][ik - 1], self.at(msk, ik))
            ml = ml / torch.maximum(out["hmlpt"], nb(out["hmlpt"])).clamp(min=5.0)
            zf = torch.maximum(oml, nb(oml))
            zdep = 0.5 * ((dep + nb(dep)) - self.e3t[0])
            raw = ((1 - zf) * za / (lim(zb, za, self.e3t, 1 / RN_SLPMAX) - eps) + zf * zdep * ml) * msk
            a = filt(lbc(raw, jp, "U"))
            a = a * (across[0](msk) + across[1](msk)) * 0.5 * (msk + kdown(msk)) * 0.5
            out[name] = lbc(a * lev, jp, nat)
        ik = (nm + 1).clamp(max=self.d.jpk)
        taper = (m.u + xm(m.u)) * (m.v + ym(m.v)) * 0.25 * m.w
        for name, back, grad, width, msk in (("wslpi", xm, gu, e["e1t"], m.u), ("wslpj", ym, gv, e["e2t"], m.v)):
            four = lambda a: back(a) + kup(a) + back(kup(a)) + a  # noqa: E731
            den = four(msk).clamp(min=eps) * width
            zbw = -0.5 / g * n2 * (prd + kup(prd) + 2)
            # just below the mixed layer: t-mask there
            za = self.at(four(grad) / den, ik) * self.at(m.t, ik)
            zb = lim(self.at(zbw, ik), za, self.e3w[:, 0, 0][ik - 1], 100.0)
            ml = za / (zb - eps) * self.at(m.t, ik)
            za = four(grad) / den * m.w
            zb = lim(zbw, za, self.e3w, 100.0)
            zf = torch.maximum(oml, kup(oml))
            zck = depw / out["hmlp"].clamp(min=10.0)
            raw = (za / (zb - eps) * (1 - zf) + zck * ml * zf) * m.w
            out[name] = lbc(filt(lbc(raw, jp, "W")) * taper * lev, jp, "W")


def _thomas(lo, di, up, rhs, mask=None):
    """tridiagonal systems along the first axis; mask multiplies each solved value before it is used above"""
    piv, f = [di[0]], [rhs[0]]
    for k in range(1, di.shape[0]):
        r = lo[k] / piv[-1]
        piv.append(di[k] - r * up[k - 1])
        f.append(rhs[k] - r * f[-1])
    x = [f[-1] / piv[-1] * (1.0 if mask is None else mask[-1])]
    for k in range(di.shape[0] - 2, -1, -1):
        x.append((f[k] - up[k] * x[-1]) / piv[k] * (1.0 if mask is None else mask[k]))
    return torch.stack(x[::-1])


def _bt_weights(n):
    """the boxcar weights of the barotropic time averages, over 0.5 n to 1.5 n sub-steps"""
    w1 = [1.0 if abs(k - n) / n < 0.5 else 0.0 for k in range(1, 3 * n + 1)]
    last = max(k for k in range(3 * n) if w1[k]) + 1
    w1 = w1[:last]
    w2 = [sum(w1[k:]) for k in range(last)]
    return [a / sum(w1) for a in w1], [a / sum(w2) for a in w2]


# The TEOS-10 polynomial of density (Roquet, Madec, McDougall and Barker, 2015, Ocean Modelling 90), with the
# coefficients NEMO uses: TEOS10[k][j][i] of s^i t^j z^k
TEOS10 = (
    ((8.0189615746e+02, 8.6672408165e+02, -1.7864682637e+03, 2.0375295546e+03, -1.2849161071e+03, 4.3227585684e+02,
      -6.0579916612e+01),
     (2.6010145068e+01, -6.5281885265e+01, 8.1770425108e+01, -5.6888046321e+01, 1.7681814114e+01, -1.9193502195),
     (-3.7074170417e+01, 6.1548258127e+01, -6.0362551501e+01, 2.9130021253e+01, -5.4723692739),
     (2.1661789529e+01, -3.3449108469e+01, 1.9717078466e+01, -3.1742946532),
     (-8.3627885467, 1.1311538584e+01, -5.3563304045),
     (5.4048723791e-01, 4.8169980163e-01),
     (-1.9083568888e-01,)),
    ((1.9681925209e+01, -4.2549998214e+01, 5.0774768218e+01, -3.0938076334e+01, 6.6051753097),
     (-1.3336301113e+01, -4.4870114575, 5.0042598061, -6.5399043664e-01),
     (6.7080479603, 3.5063081279, -1.8795372996),
     (-2.4649669534, -5.5077101279e-01),
     (5.5927935970e-01,)),
    ((2.0660924175, -4.9527603989, 2.5019633244),
     (2.0564311499, -2.1311365518e-01),
     (-1.2419983026,)),
    ((-2.3342758797e-02, -1.8507636718e-02),
     (3.7969820455e-01,)),
)


def exact(case, seed, device="cuda"):
    out = []
    for q, g in enumerate(_members(case)):
        d = _grid(nemo_hip.get(), g)[1] if device == "cuda" else _domain(g)
        X = Exact(case, d, _inputs(case, g, d, int(seed) * 64 + q, device), device)
        r = getattr(X, "step" if case["kind"] == "ensemble" else case["kind"])()
        del X
        names = r.keys() if case["kind"] == "adjoint" else _out_names(case)
        out.append({k: (None if r[k] is None else r[k].reshape(-1)) for k in names})
    return out if case["kind"] == "ensemble" else out[0]
