"""The momentum kernels where a workgroup takes whole columns, and both
components of them: eagerly from 512 workgroups (k_step_dyn1 with its sums, the
f-point tiles of EEN and EET among them) and 1024 (the column solves), and in
a plan at any size.  Against the oracle with the parity tests' 1e-12; the
plan against the eager calls bit for bit."""
import numpy as np
import pytest

from nemo_hip import abi, configs
from oracle.oracle import Oracle
from test_gpu_ensemble import OPTS, _state, _stepper
from test_gpu_parity import SPG_OUT, Env, check, dev, host, spg_fields, sync
from test_gpu_step import nan_like, oracle_dyn_step

torch = pytest.importorskip("torch")


@pytest.mark.gpu
@pytest.mark.parametrize("vor,jperio", [("een", 0), ("een", 7), ("eet", 1), ("ene", 0)])
def test_step_dyn_and_dyn_zdf_of_a_wide_domain(hip, vor, jperio):
    e = Env.__new__(Env)
    d = configs.basin(1030, 243, 6, seed=12, jperio=jperio, opts={"nvor_scheme": abi.VOR_NAMES[vor]})
    e.d, e.S, e.o = d, configs.make_state(d, seed=13), Oracle(d)
    hip.register(d)
    e.s3, e.s2 = (d.jpi, d.jpj, d.jpk), (d.jpi, d.jpj)
    S = e.S
    ua, va = e.c("ua"), e.c("va")
    args = [S[n] for n in ("avm", "rCdU_bot", "ua_b", "va_b", "utau", "utau_b", "vtau", "vtau_b")]
    gu, gv = dev(ua), dev(va)
    e.o.dyn_zdf(7, S["ub"], S["vb"], ua, va, *args)
    hip.dyn_zdf(7, dev(S["ub"]), dev(S["vb"]), gu, gv, *[dev(a) for a in args])
    sync(hip)
    check(host(gu, e.s3), ua, what="dyn_zdf ua")
    check(host(gv, e.s3), va, what="dyn_zdf va")
    Fo = spg_fields(e)
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
@pytest.mark.parametrize("vor", ["een", "eet"])
def test_a_plan_of_small_members_equals_the_eager_calls(hip, vor):
    members = [(40, 30, 12, 0, 3), (66, 31, 10, 0, 5), (44, 26, 9, 7, 8)]
    ctxs, eager, planned, plan = [], [], [], None
    try:
        for jpi, jpj, jpk, jperio, seed in members:
            ctxs.append(hip.context_create())
            hip.context_select(ctxs[-1])
            d = configs.basin(jpi, jpj, jpk, seed=seed, jperio=jperio, opts=dict(OPTS, nvor_scheme=abi.VOR_NAMES[vor]))
            hip.register(d)
            eager.append(_stepper(hip, d, seed + 100))
            planned.append(_stepper(hip, d, seed + 100))
        for kt in (1, 2):
            for c, a, b in zip(ctxs, eager, planned):
                hip.context_select(c)
                a.step(kt)
                b.step(kt)
        hip.sync()
        hip.plan_begin()
        for c, b in zip(ctxs, planned):
            hip.context_select(c)
            b.step(3)
        plan = hip.plan_end()
        for kt in (3, 4):
            for c, a in zip(ctxs, eager):
                hip.context_select(c)
                a.step(kt)
            hip.plan_launch(plan)
            hip.sync()
            torch.cuda.synchronize()
            for m, (a, b) in enumerate(zip(eager, planned)):
                sa, sb = _state(a), _state(b)
                for k in sa:
                    assert np.all(np.isfinite(sa[k])) and np.array_equal(sa[k], sb[k]), f"member {m} {k} kt {kt}"
    finally:
        if plan is not None:
            hip.plan_free(plan)
        hip.context_select(0)
        del eager, planned
        for c in ctxs:
            hip.context_destroy(c)
