"""The limiter's stop at the bottom (FctDry: a word on the device holds the
number of the last call whose transports were not zero on land) over calls that
follow one another on one domain: masked and unmasked transports in turn, a
recorded call replayed with eager calls between, the fused tracer step with
unmasked velocities, FP32 storage.  FP64 against the oracle with the parity
tests' 1e-12; FP32 storage against the one-kernel form of the chain (switch
fct_fused), which marches every level and gives the same bits."""
import numpy as np
import pytest

from nemo_hip import configs
from oracle.oracle import Oracle
from test_gpu_parity import check, dev, host, sync

torch = pytest.importorskip("torch")

ORDER = "MUMMUUM"              # masked, unmasked


def setup(hip, jpk=31):
    d = configs.basin(92, 40, jpk, seed=jpk, opts={"neuler": 1})
    hip.register(d)
    return d, configs.make_state(d, seed=4), np.random.default_rng(8)


def spoil(a, rng):
    """values where a masked field is zero: on land, and on faces of land"""
    return np.asfortranarray(np.where(a == 0.0, a.std() * rng.standard_normal(a.shape), a))


def transports(d, S, rng):
    z = [np.zeros((d.jpi, d.jpj, d.jpk), order="F") for _ in range(3)]
    Oracle(d).tra_adv_trp(S["un"], S["vn"], S["wn"], *z)
    return {"M": z, "U": [spoil(a, rng) for a in z]}


@pytest.mark.gpu
@pytest.mark.parametrize("kn", [2, 4])
def test_calls_in_turn(hip, kn):
    d, S, rng = setup(hip)
    trp, s4, p2dt, o = transports(d, S, rng), (d.jpi, d.jpj, d.jpk, 2), 2.0 * d.opts["rdt"], Oracle(d)
    want = {}
    for m, z in trp.items():
        want[m] = S["tsa"].copy(order="F")
        o.tra_adv_fct(3, 1, "TRA", p2dt, *z, S["tsb"], S["tsn"], want[m], 2, kn, kn)
    for q, m in enumerate(ORDER):
        ta = dev(S["tsa"])
        hip.tra_adv_fct(3, 1, "TRA", p2dt, *(dev(a) for a in trp[m]), dev(S["tsb"]), dev(S["tsn"]), ta, 2, kn, kn)
        sync(hip)
        check(host(ta, s4), want[m], what=f"call {q} {m}")


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["graph", "plan"])
def test_a_recorded_call_replayed(hip, how):
    d, S, rng = setup(hip)
    trp, s4, p2dt, o = transports(d, S, rng), (d.jpi, d.jpj, d.jpk, 2), 2.0 * d.opts["rdt"], Oracle(d)
    want = {}
    for m, z in trp.items():
        want[m] = S["tsa"].copy(order="F")
        o.tra_adv_fct(3, 1, "TRA", p2dt, *z, S["tsb"], S["tsn"], want[m], 2, 4, 4)
    dz = {m: [dev(a) for a in z] for m, z in trp.items()}
    buf, ta, ta0, tb, tn = [torch.empty_like(a) for a in dz["M"]], dev(S["tsa"]), dev(S["tsa"]), dev(S["tsb"]), dev(S["tsn"])
    begin, end, launch, free = ((hip.graph_begin, hip.graph_end, hip.graph_launch, hip.graph_free) if how == "graph" else
                                (hip.plan_begin, hip.plan_end, hip.plan_launch, hip.plan_free))
    begin()
    hip.tra_adv_fct(3, 1, "TRA", p2dt, *buf, tb, tn, ta, 2, 4, 4)
    g = end()
    try:
        for q, m in enumerate(ORDER):
            for b, a in zip(buf, dz[m]):
                b.copy_(a)
            ta.copy_(ta0)
            torch.cuda.synchronize()
            launch(g)
            sync(hip)
            check(host(ta, s4), want[m], what=f"replay {q} {m}")
            if q % 2:                       # an eager call of the other kind
                e, n = ta0.clone(), "U" if m == "M" else "M"
                hip.tra_adv_fct(3, 1, "TRA", p2dt, *dz[n], tb, tn, e, 2, 4, 4)
                sync(hip)
                check(host(e, s4), want[n], what=f"eager {q} {n}")
    finally:
        free(g)


@pytest.mark.gpu
@pytest.mark.parametrize("kn", [2, 4])
@pytest.mark.parametrize("sp", [False, True], ids=["fp64", "fp32"])
def test_step_tra_with_unmasked_velocities(hip, sp, kn):
    d, S, rng = setup(hip)
    dt = torch.float32 if sp else torch.float64
    vel = {"M": [S[n] for n in ("un", "vn", "wn")], "U": [spoil(S[n], rng) for n in ("un", "vn", "wn")]}
    f = {n: dev(S[n], dt) for n in ("tsb", "tsn", "ahtu", "ahtv", "uslp", "vslp", "wslpi", "wslpj", "avt")}
    n3 = d.jpi * d.jpj * d.jpk

    def step(m):
        tsa, ah, akz = (torch.zeros(n * n3, dtype=dt, device="cuda") for n in (2, 1, 1))
        hip.step_tra(3, *(dev(a, dt) for a in vel[m]), f["tsb"], f["tsn"], tsa, kn, kn, f["ahtu"], f["ahtv"], f["uslp"],
                     f["vslp"], f["wslpi"], f["wslpj"], ah, akz, f["avt"], sp=sp)
        sync(hip)
        return tsa

    was = hip.tune_get("fct_fused")
    try:
        hip.tune_set("fct_fused", 1)
        want = {m: step(m) for m in vel}
        hip.tune_set("fct_fused", 0)
        assert not torch.equal(want["M"], want["U"])
        for q, m in enumerate(ORDER):
            assert torch.equal(step(m), want[m]), f"call {q} {m}"
    finally:
        hip.tune_set("fct_fused", was)
