"""dyn_spg_ts's blocks of sub-steps (k_spg_blk) against the oracle at the
sizes where a region's edges can go wrong: a domain that is exactly one region
(32 points), one point more, sides of several regions with a remainder, cyclic
sides shorter than a region's halo, and both sides cyclic.  Two calls (Euler
start, leapfrog) per case; the bar is the parity tests' 1e-12."""
import numpy as np
import pytest

from nemo_hip import abi, configs
from oracle.oracle import Oracle
from test_gpu_parity import SPG_OUT, Env, check, dev, host, spg_fields, sync

torch = pytest.importorskip("torch")

SIZES = [(32, 32, 0), (33, 31, 0), (34, 70, 0), (131, 45, 0), (8, 9, 7), (5, 40, 1), (40, 6, 2), (65, 67, 7),
         (33, 100, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("jpi,jpj,jperio", SIZES)
@pytest.mark.parametrize("scheme", ["ene", "ens", "mix", "eet", "een"])
def test_blocks_against_oracle(hip, jpi, jpj, jperio, scheme):
    opts = {"nvor_scheme": abi.VOR_NAMES[scheme], "rdt": 600.0}
    e = Env(hip, "gyre", opts=opts)
    d = (configs.basin(jpi, jpj, 5, seed=jpi + jpj, jperio=jperio, opts=opts) if min(jpi, jpj) >= 30 else
         configs.gyre_like(jpi, jpj, 5, jperio=jperio, opts=opts))
    hip.register(d)
    e.d, e.S, e.o = d, configs.make_state(d, seed=7), Oracle(d)
    e.s3, e.s2 = (d.jpi, d.jpj, d.jpk), (d.jpi, d.jpj)
    Fo = spg_fields(e)
    Fd = {k: dev(v) for k, v in Fo.items()}
    for kt in (1, 2):
        e.o.dyn_spg_ts(kt, Fo)
        hip.dyn_spg_ts(kt, Fd)
        sync(hip)
        for k in ["ua", "va", "un", "vn", "ub2_b", "vb2_b", "un_bf", "vn_bf"] + SPG_OUT:
            shape = e.s3 if k in ("ua", "va", "un", "vn") else e.s2
            check(host(Fd[k], shape), Fo[k], what=f"{jpi}x{jpj} jperio {jperio} {scheme} kt={kt} {k}")
            assert np.isfinite(Fo[k]).all()
