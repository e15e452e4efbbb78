"""ldf_slp and dyn_ldf_lap at the edges of their regions against the oracle:
domains one tile wide, one point more, several tiles with a remainder, cyclic
sides shorter than a region, level counts around the chunks of a march.  The
bar is the parity tests' 1e-12 (the operations are the oracle's, in its order)."""
import numpy as np
import pytest

from nemo_hip import abi, configs
from oracle.oracle import Oracle
from test_gpu_parity import Env, check, dev, host, sync

torch = pytest.importorskip("torch")

SIZES = [(30, 14, 9, 0), (31, 15, 10, 0), (92, 40, 30, 0), (9, 8, 5, 7), (36, 11, 27, 1), (12, 60, 28, 2), (64, 47, 75, 7)]


def grid(jpi, jpj, jpk, jperio):
    if min(jpi, jpj) >= 30:
        return configs.basin(jpi, jpj, jpk, seed=jpi + jpk, jperio=jperio)
    return configs.gyre_like(jpi, jpj, jpk, jperio=jperio)


@pytest.mark.gpu
@pytest.mark.parametrize("jpi,jpj,jpk,jperio", SIZES)
def test_slopes_and_viscosity_at_region_edges(hip, jpi, jpj, jpk, jperio):
    e = Env(hip, "gyre")
    d = grid(jpi, jpj, jpk, jperio)
    hip.register(d)
    o, S = Oracle(d), configs.make_state(d, seed=5)
    s3, s2 = (d.jpi, d.jpj, d.jpk), (d.jpi, d.jpj)
    rng = np.random.default_rng(3)
    ts = S["tsb"].copy(order="F")
    ts[..., 0] += 2.0 * rng.standard_normal(s2)[:, :, None]      # lateral contrasts: slopes below and at the limit
    eos = abi.seos()
    o.eos_register(eos)
    gdept, gdepw = configs.depths(d)
    pab, n2, rhd = np.zeros(s3 + (2,), order="F"), np.zeros(s3, order="F"), np.zeros(s3, order="F")
    o.rab_3d(ts, pab, gdept)
    o.bn2(ts, pab, n2, gdept, gdepw)
    o.eos_insitu(ts, rhd, gdept)
    nmln, hmlp, hmlpt = o.zdf_mxl(2, n2, gdept, gdepw, configs.nlb10(d))
    want = [np.asfortranarray(rng.standard_normal(s3)) for _ in range(4)]
    got = [dev(a) for a in want]
    o.ldf_slp(2, rhd, n2, gdept, gdepw, nmln, hmlp, hmlpt, 0.01, *want)
    hip.ldf_slp(2, dev(rhd), dev(n2), dev(gdept), dev(gdepw), dev(nmln, torch.int32), dev(hmlp), dev(hmlpt), 0.01, *got)
    u, v, ua, va, ahmt, ahmf = (np.asfortranarray(rng.standard_normal(s3)) for _ in range(6))
    dua, dva = dev(ua), dev(va)
    o.dyn_ldf_lap(2, u, v, ua, va, 1, ahmt, ahmf)
    hip.dyn_ldf_lap(2, dev(u), dev(v), dua, dva, 1, dev(ahmt), dev(ahmf))
    sync(hip)
    for n, w, g in zip(("uslp", "vslp", "wslpi", "wslpj", "ua", "va"), want + [ua, va], got + [dua, dva]):
        check(host(g, s3), w, what=f"{jpi}x{jpj}x{jpk} jperio {jperio} {n}")
