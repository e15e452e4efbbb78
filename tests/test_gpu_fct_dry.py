"""tra_adv_fct where its kernels split or shorten their work, against the
oracle: small grids whose levels are shared out over workgroups (remainders,
single chunks), cyclic sides, one to three tracers, both orders, and
transports that are zero on land (the limiter stops at the bottom) or not (it
may not).  The bar is the parity tests' 1e-12."""
import numpy as np
import pytest

from nemo_hip import configs
from oracle.oracle import Oracle
from test_gpu_parity import check, dev, host, sync

torch = pytest.importorskip("torch")

SIZES = [(30, 14, 9, 0, 2), (31, 15, 10, 0, 1), (92, 40, 31, 0, 3), (9, 8, 5, 7, 2), (36, 33, 27, 1, 3), (66, 47, 75, 0, 2)]


@pytest.mark.gpu
@pytest.mark.parametrize("masked", [True, False])
@pytest.mark.parametrize("orders", [(2, 2), (4, 4)])
@pytest.mark.parametrize("jpi,jpj,jpk,jperio,ntr", SIZES)
def test_fct_chunks_and_dry_levels(hip, jpi, jpj, jpk, jperio, ntr, orders, masked):
    if min(jpi, jpj) >= 30:
        d = configs.basin(jpi, jpj, jpk, seed=jpi + jpk, jperio=jperio)
    else:
        d = configs.gyre_like(jpi, jpj, jpk, jperio=jperio)
    hip.register(d)
    o, S = Oracle(d), configs.make_state(d, seed=4)
    s3 = (d.jpi, d.jpj, d.jpk)
    rng = np.random.default_rng(8)
    z = [np.zeros(s3, order="F") for _ in range(3)]
    o.tra_adv_trp(S["un"], S["vn"], S["wn"], *z)
    if not masked:
        z = [np.asfortranarray(np.where(a == 0.0, a.std() * rng.standard_normal(s3), a)) for a in z]
    tb, tn, ta = (np.asfortranarray(np.stack([S[n][..., t % 2] * (1.0 + 0.1 * t) for t in range(ntr)], axis=-1))
                  for n in ("tsb", "tsn", "tsa"))
    got, p2dt = dev(ta), 2.0 * d.opts["rdt"]
    hip.tra_adv_fct(3, 1, "TRA", p2dt, *(dev(a) for a in z), dev(tb), dev(tn), got, ntr, *orders)
    o.tra_adv_fct(3, 1, "TRA", p2dt, *z, tb, tn, ta, ntr, *orders)
    sync(hip)
    check(host(got, s3 + (ntr,)), ta, what=f"{jpi}x{jpj}x{jpk} jperio {jperio} {orders} masked {masked}")
