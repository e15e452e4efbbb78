"""The density kernels on domains on either side of the share of dry waves
from which they test their waves for land (an eighth): rows of a closed basin
turned to land, from none to all but one.  FP64 against the oracle with the
parity tests' 1e-12, FP32 storage with the 1e-6 of its tests."""
import numpy as np
import pytest

from nemo_hip import abi, configs
from oracle.oracle import Oracle
from test_gpu_parity import sync
from test_gpu_phys import cmp, g, host, rnd, tracers

torch = pytest.importorskip("torch")


class E:
    pass


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [0, 2, 3, 16, 31])      # of 34, two of them the ring: 2/34 to 33/34 dry
@pytest.mark.parametrize("scheme", ["teos10", "eos80", "seos"])
@pytest.mark.parametrize("sp", [False, True])
def test_land_share(hip, rows, scheme, sp):
    d = configs.gyre_like(130, 34, 9)
    d.arrays["k_top"][:, 1:1 + rows] = 0
    d.arrays["k_bot"][:, 1:1 + rows] = 0
    hip.register(d)
    e = E()
    e.d, e.o, e.s3, e.s4 = d, Oracle(d), (d.jpi, d.jpj, d.jpk), (d.jpi, d.jpj, d.jpk, 2)
    par = getattr(abi, scheme)()
    hip.eos_register(par)
    e.o.eos_register(par)
    rng = np.random.default_rng(rows)
    ts, (z, _) = tracers(rng, e, sp), configs.depths(d)
    if sp:
        z = np.asfortranarray(z.astype(np.float32).astype(np.float64))
    prd, pab = rnd(rng, e.s3, sp), rnd(rng, e.s4, sp)
    want, want2, wantp, wab = prd.copy(order="F"), prd.copy(order="F"), prd.copy(order="F"), pab.copy(order="F")
    got, got2, gotp, gab = g(prd, sp), g(prd, sp), g(prd, sp), g(pab, sp)
    e.o.eos_insitu(ts, want, z)
    e.o.eos_insitu_pot(ts, want2, wantp, z)
    e.o.rab_3d(ts, wab, z)
    hip.eos_insitu(g(ts, sp), got, g(z, sp), sp=sp)
    hip.eos_insitu_pot(g(ts, sp), got2, gotp, g(z, sp), sp=sp)
    hip.rab_3d(g(ts, sp), gab, g(z, sp), sp=sp)
    sync(hip)
    for n, a, w in (("rhd", got, want), ("rhd of pot", got2, want2), ("rhop", gotp, wantp)):
        cmp(host(a, e.s3), w, sp, n)
    cmp(host(gab, e.s4), wab, sp, "rab")
