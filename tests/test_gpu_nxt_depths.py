"""The closure kernels at the edges of their batches of levels and of the
columns that dyn_nxt keeps in registers, with scale factors that are
horizontally uniform or not, closed and cyclic sides: FP64 against the oracle
with the parity tests' 1e-12."""
import numpy as np
import pytest

from nemo_hip import configs
from oracle.oracle import Oracle
from test_gpu_nxt import DYN2, DYN3, DYN_NXT_OPTS, Fields, dyn_nxt_pair
from test_gpu_parity import Env, check, host, sync

torch = pytest.importorskip("torch")


@pytest.mark.gpu
@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("jpk,jperio,opt", [(3, 0, "ts_fw"), (9, 1, "ts_centred"), (10, 7, "ts_fw"), (33, 0, "ts_fw"),
                                            (34, 1, "no_ts"), (49, 2, "ts_fw"), (50, 0, "ts_centred"),
                                            (81, 7, "ts_fw"), (82, 1, "ts_fw"), (91, 0, "ts_centred")])
def test_closure_at_batch_edges(hip, jpk, jperio, opt, uniform):
    d = configs.basin(37, 26, jpk, seed=jpk, jperio=jperio, opts=DYN_NXT_OPTS[opt])
    if not uniform:
        rng = np.random.default_rng(jpk)
        for n in ("e3t_n", "e3u_n", "e3v_n"):
            d.arrays[n] *= 1.0 + 0.2 * rng.random(d.arrays[n].shape)
    hip.register(d)
    e = Env.__new__(Env)
    e.d, e.S, e.o = d, configs.make_state(d, seed=2), Oracle(d)
    s3, s2 = (d.jpi, d.jpj, d.jpk), (d.jpi, d.jpj)
    shapes = {n: s3 for n in DYN3 + ("hdivn", "wn")}
    shapes.update({n: s2 for n in DYN2 + ("sshb", "emp_b", "emp", "ssha")})
    f = Fields(e, 70 + jpk, False, **shapes)
    o, g = ({n: fn(n) for n in ("un", "vn", "hdivn", "wn", "sshb", "emp_b", "emp", "ssha")} for fn in (f.o, f.g))
    e.o.div_hor(3, o["un"], o["vn"], o["hdivn"])
    hip.div_hor(3, g["un"], g["vn"], g["hdivn"])
    sync(hip)
    check(host(g["hdivn"], s3), o["hdivn"], what="div_hor")
    for h, a in ((e.o, o), (hip, g)):
        h.ssh_nxt(3, *[a[n] for n in ("un", "vn", "hdivn", "sshb", "emp_b", "emp", "ssha")])
        h.wzv(3, a["hdivn"], a["wn"])
    sync(hip)
    for n in ("hdivn", "wn", "ssha"):
        check(host(g[n], s2 if n == "ssha" else s3), o[n], what=n)
    for kt in (1, 6):
        o, g = dyn_nxt_pair(hip, e, f, kt, False)
        for n in DYN3 + ("ub_b", "vb_b", "un_b", "vn_b"):
            check(host(g[n], s2 if n.endswith("_b") else s3), o[n], what=f"dyn_nxt kt={kt} {n}")
