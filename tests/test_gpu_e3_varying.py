"""The kernels that have one form for horizontally uniform scale factors (a
scalar load per level) and one for scale factors that vary over the domain:
the varying form against the oracle, all seven e3 arrays perturbed point by
point, at level counts around the 4-level segments of the column solves,
closed and cyclic sides.  FP64 with the parity tests' 1e-12 (the operations
are the oracle's, in its order); FP32 storage as fused against separate
calls, which round alike and so give the same bits."""
import numpy as np
import pytest

from nemo_hip import abi, configs
from oracle.oracle import Oracle
from test_gpu_parity import SPG_OUT, Env, check, dev, host, spg_fields, sync
from test_gpu_step import nan_like, oracle_dyn_step, oracle_tra_step, r2dt

torch = pytest.importorskip("torch")

# (jpk, jperio): one and two segments with every remainder, and a deep column
LEVELS = [(4, 0), (5, 1), (6, 7), (7, 0), (8, 2), (9, 1), (31, 0), (75, 7)]


def env(hip, jpk, jperio, opts=None):
    e = Env.__new__(Env)
    d = configs.basin(38, 29, jpk, seed=jpk, jperio=jperio, opts=opts)
    rng = np.random.default_rng(100 + jpk)
    for n in ("e3t_n", "e3u_n", "e3v_n", "e3w_n", "e3f_n", "e3uw_n", "e3vw_n"):
        d.arrays[n] = np.asfortranarray(d.arrays[n] * (1.0 + 0.2 * rng.random(d.arrays[n].shape)))
    e.d, e.S, e.o, e.h = d, configs.make_state(d, seed=jpk + 1), Oracle(d), hip
    hip.register(d)
    e.s3, e.s4, e.s2 = (d.jpi, d.jpj, d.jpk), (d.jpi, d.jpj, d.jpk, 2), (d.jpi, d.jpj)
    return e


@pytest.mark.gpu
@pytest.mark.parametrize("jpk,jperio", LEVELS)
@pytest.mark.parametrize("orders", [(2, 2), (4, 4)])
def test_tra_adv_fct(hip, jpk, jperio, orders):
    e = env(hip, jpk, jperio)
    S, z, want, p2dt = e.S, [np.zeros(e.s3, order="F") for _ in range(3)], e.c("tsa"), 2.0 * e.d.opts["rdt"]
    e.o.tra_adv_trp(S["un"], S["vn"], S["wn"], *z)
    e.o.tra_adv_fct(3, 1, "TRA", p2dt, *z, S["tsb"], S["tsn"], want, 2, *orders)
    ta = dev(S["tsa"])
    hip.tra_adv_fct(3, 1, "TRA", p2dt, *(dev(a) for a in z), dev(S["tsb"]), dev(S["tsn"]), ta, 2, *orders)
    sync(hip)
    check(host(ta, e.s4), want, what="tsa")


@pytest.mark.gpu
@pytest.mark.parametrize("jpk,jperio", LEVELS)
@pytest.mark.parametrize("lap,msc,ntr", [(1, 0, 2), (1, 1, 1), (0, 0, 1), (0, 1, 2)])
def test_tra_ldf_iso_both_passes(hip, jpk, jperio, lap, msc, ntr):
    e = env(hip, jpk, jperio, opts={"ln_traldf_lap": lap, "ln_traldf_msc": msc})
    S, tb = e.S, np.asfortranarray(e.S["tsb"][..., :ntr])
    names = ("uslp", "vslp", "wslpi", "wslpj")
    ah_o, akz_o = np.zeros(e.s3, order="F"), np.zeros(e.s3, order="F")
    ah, akz = dev(ah_o), dev(akz_o)
    s4 = e.s3 + (ntr,)
    lap_o, lap_d = np.zeros(s4, order="F"), dev(np.zeros(s4))
    for kpass in ((1,) if lap else (1, 2)):            # the bilaplacian's second pass acts on the first one's result
        b = tb if kpass == 1 else lap_o
        want = np.zeros(s4, order="F") if not lap and kpass == 1 else np.asfortranarray(S["tsa"][..., :ntr].copy())
        got = dev(want)
        e.o.tra_ldf_iso(5, 1, "TRA", S["ahtu"], S["ahtv"], b, tb, want, ntr, kpass, *(S[n] for n in names), ah_o, akz_o)
        hip.tra_ldf_iso(5, 1, "TRA", dev(S["ahtu"]), dev(S["ahtv"]), dev(b), dev(tb), got, ntr, kpass,
                        *(dev(S[n]) for n in names), ah, akz)
        sync(hip)
        check(host(got, s4), want, what=f"pass {kpass}")
        check(host(ah, e.s3), ah_o, what="ah_wslp2")
        check(host(akz, e.s3), akz_o, what="akz")
        if not lap:
            lap_o = want


@pytest.mark.gpu
@pytest.mark.parametrize("jpk,jperio", LEVELS)
@pytest.mark.parametrize("ntr,slp", [(1, 0), (2, 1), (2, 0), (3, 1)])
def test_tra_zdf(hip, jpk, jperio, ntr, slp):
    e = env(hip, jpk, jperio)
    S = e.S
    tb, ta = (np.asfortranarray(np.stack([S[n][..., t % 2] for t in range(ntr)], axis=-1)) for n in ("tsb", "tsa"))
    ah, got = np.asfortranarray(np.abs(S["wslpi"])), dev(ta)
    e.o.tra_zdf_imp(4, 1, "TRC", 3600.0, tb, ta, ntr, S["avt"], S["avt"], slp, ah, ah)
    hip.tra_zdf_imp(4, 1, "TRC", 3600.0, dev(tb), got, ntr, dev(S["avt"]), dev(S["avt"]), slp, dev(ah), dev(ah))
    sync(hip)
    check(host(got, e.s3 + (ntr,)), ta, what="tra_zdf_imp")


@pytest.mark.gpu
@pytest.mark.parametrize("jpk,jperio", LEVELS)
def test_dyn_zdf(hip, jpk, jperio):
    e = env(hip, jpk, jperio)
    S, ua, va = e.S, e.c("ua"), e.c("va")
    args = [S[n] for n in ("avm", "rCdU_bot", "ua_b", "va_b", "utau", "utau_b", "vtau", "vtau_b")]
    gu, gv = dev(ua), dev(va)
    e.o.dyn_zdf(7, S["ub"], S["vb"], ua, va, *args)
    hip.dyn_zdf(7, dev(S["ub"]), dev(S["vb"]), gu, gv, *[dev(a) for a in args])
    sync(hip)
    check(host(gu, e.s3), ua, what="ua")
    check(host(gv, e.s3), va, what="va")


@pytest.mark.gpu
@pytest.mark.parametrize("jpk,jperio", LEVELS)
@pytest.mark.parametrize("vor", ["ene", "een", "eet"])
def test_step_dyn(hip, jpk, jperio, vor):
    e = env(hip, jpk, jperio, opts={"nvor_scheme": abi.VOR_NAMES[vor]})
    Fo, S = spg_fields(e), e.S
    Fd = {k: dev(v) for k, v in Fo.items()}
    Fd["ua"], Fd["va"] = nan_like(Fd["ua"]), nan_like(Fd["va"])
    args = [dev(S[n]) for n in ("ub", "vb", "wn", "avm", "utau_b", "vtau_b")]
    for kt in (1, 2):
        oracle_dyn_step(e, kt, Fo)
        hip.step_dyn(kt, *args, Fd)
        sync(hip)
        for k in ["ua", "va", "un", "vn"] + SPG_OUT:
            check(host(Fd[k], e.s3 if k in ("ua", "va", "un", "vn") else e.s2), Fo[k], what=f"kt={kt} {k}")


@pytest.mark.gpu
@pytest.mark.parametrize("jpk,jperio", LEVELS)
@pytest.mark.parametrize("orders,msc", [((4, 4), 0), ((2, 2), 1)])
def test_step_tra(hip, jpk, jperio, orders, msc):
    e = env(hip, jpk, jperio, opts={"ln_traldf_msc": msc})
    ah, akz = np.zeros(e.s3, order="F"), np.zeros(e.s3, order="F")
    f = {n: dev(e.S[n]) for n in ("un", "vn", "wn", "tsb", "tsn", "ahtu", "ahtv", "uslp", "vslp", "wslpi", "wslpj", "avt")}
    gah, gakz, tsa = dev(ah), dev(akz), dev(np.full(e.s4, np.nan))
    want = oracle_tra_step(e, 2, orders, ah, akz)
    hip.step_tra(2, *(f[n] for n in ("un", "vn", "wn", "tsb", "tsn")), tsa, *orders,
                 *(f[n] for n in ("ahtu", "ahtv", "uslp", "vslp", "wslpi", "wslpj")), gah, gakz, f["avt"])
    sync(hip)
    check(host(tsa, e.s4), want, what="tsa")


@pytest.mark.gpu
@pytest.mark.parametrize("jpk,jperio", LEVELS)
def test_slopes_and_lateral_viscosity(hip, jpk, jperio):
    e = env(hip, jpk, jperio)
    d, o, rng = e.d, e.o, np.random.default_rng(3)
    ts = e.c("tsb")
    ts[..., 0] += 2.0 * rng.standard_normal(e.s2)[:, :, None]      # lateral contrasts: slopes below and at the limit
    o.eos_register(abi.seos())
    gdept, gdepw = configs.depths(d)
    pab, n2, rhd = np.zeros(e.s4, order="F"), np.zeros(e.s3, order="F"), np.zeros(e.s3, order="F")
    o.rab_3d(ts, pab, gdept)
    o.bn2(ts, pab, n2, gdept, gdepw)
    o.eos_insitu(ts, rhd, gdept)
    nmln, hmlp, hmlpt = o.zdf_mxl(2, n2, gdept, gdepw, configs.nlb10(d))
    want = [np.asfortranarray(rng.standard_normal(e.s3)) for _ in range(4)]
    got = [dev(a) for a in want]
    o.ldf_slp(2, rhd, n2, gdept, gdepw, nmln, hmlp, hmlpt, 0.01, *want)
    hip.ldf_slp(2, dev(rhd), dev(n2), dev(gdept), dev(gdepw), dev(nmln, torch.int32), dev(hmlp), dev(hmlpt), 0.01, *got)
    u, v, ua, va, ahmt, ahmf = (np.asfortranarray(rng.standard_normal(e.s3)) for _ in range(6))
    gu, gv = dev(ua), dev(va)
    o.dyn_ldf_lap(2, u, v, ua, va, 1, ahmt, ahmf)
    hip.dyn_ldf_lap(2, dev(u), dev(v), gu, gv, 1, dev(ahmt), dev(ahmf))
    sync(hip)
    for n, w, g in zip(("uslp", "vslp", "wslpi", "wslpj", "ua", "va"), want + [ua, va], got + [gu, gv]):
        check(host(g, e.s3), w, what=n)


@pytest.mark.gpu
@pytest.mark.parametrize("jpk,jperio", [(9, 0), (31, 7)])
def test_fp32_fused_equals_separate_calls(hip, jpk, jperio):
    e = env(hip, jpk, jperio)
    S = e.S
    f = {n: dev(S[n], torch.float32) for n in ("un", "vn", "wn", "ub", "vb", "avm", "tsb", "tsn", "ahtu", "ahtv", "uslp",
                                               "vslp", "wslpi", "wslpj", "avt")}
    z = lambda n=1: torch.zeros(n * e.d.jpi * e.d.jpj * e.d.jpk, dtype=torch.float32, device="cuda")  # noqa: E731
    # tracers
    trp, ah, akz, tsa, ah2, akz2, tsa2 = [z() for _ in range(3)], z(), z(), z(2), z(), z(), nan_like(z(2))
    slp = [f[n] for n in ("uslp", "vslp", "wslpi", "wslpj")]
    hip.tra_adv_trp(f["un"], f["vn"], f["wn"], *trp, sp=True)
    hip.tra_adv_fct(2, 1, "TRA", r2dt(e.d, 2), *trp, f["tsb"], f["tsn"], tsa, 2, 4, 4, sp=True)
    hip.tra_ldf_iso(2, 1, "TRA", f["ahtu"], f["ahtv"], f["tsb"], f["tsb"], tsa, 2, 1, *slp, ah, akz, sp=True)
    hip.tra_zdf(2, f["tsb"], tsa, f["avt"], f["avt"], 1, ah, akz, sp=True)
    hip.step_tra(2, f["un"], f["vn"], f["wn"], f["tsb"], f["tsn"], tsa2, 4, 4, f["ahtu"], f["ahtv"], *slp, ah2, akz2,
                 f["avt"], sp=True)
    # momentum
    base = spg_fields(e)
    Fa = {k: (f[k].clone() if k in ("un", "vn") else dev(v)) for k, v in base.items()}
    Fb = {k: v.clone() for k, v in Fa.items()}
    Fa["ua"], Fa["va"], Fb["ua"], Fb["va"] = z(), z(), nan_like(z()), nan_like(z())
    two = {n: dev(S[n]) for n in ("utau_b", "vtau_b")}
    torch.cuda.synchronize()
    hip.dyn_adv(2, Fa["un"], Fa["vn"], f["wn"], Fa["ua"], Fa["va"], sp=True)
    hip.dyn_vor(2, Fa["un"], Fa["vn"], Fa["ua"], Fa["va"], sp=True)
    hip.dyn_spg_ts(2, Fa, sp=True)
    hip.dyn_zdf(2, f["ub"], f["vb"], Fa["ua"], Fa["va"], f["avm"], Fa["rCdU_bot"], Fa["ua_b"], Fa["va_b"], Fa["utau"],
                two["utau_b"], Fa["vtau"], two["vtau_b"], sp=True)
    hip.step_dyn(2, f["ub"], f["vb"], f["wn"], f["avm"], two["utau_b"], two["vtau_b"], Fb, sp=True)
    sync(hip)
    assert torch.equal(tsa, tsa2) and torch.isfinite(tsa).all()
    for k in ["ua", "va", "un", "vn"] + SPG_OUT:
        assert torch.equal(Fa[k], Fb[k]) and torch.isfinite(Fa[k]).all(), k
