"""dyn_vor and dyn_adv where their levels are shared out over workgroups and at
the edges of the EEN/EET f-point tiles (64 x 4 cells), against the oracle:
grids one cell short of a tile, a tile, one cell more; one chunk and several;
cyclic sides; scale factors that vary.  The bar is the parity tests' 1e-12."""
import numpy as np
import pytest

from nemo_hip import abi, configs
from oracle.oracle import Oracle
from test_gpu_parity import check, dev, host, sync

torch = pytest.importorskip("torch")

SIZES = [(65, 29, 4, 0), (66, 30, 6, 1), (67, 31, 12, 7), (130, 33, 31, 2), (650, 210, 6, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("scheme", ["een", "eet", "ene", "ent"])
@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("jpi,jpj,jpk,jperio", SIZES)
def test_vorticity_and_advection_at_tile_edges(hip, jpi, jpj, jpk, jperio, uniform, scheme):
    d = configs.basin(jpi, jpj, jpk, seed=jpi + jpk, jperio=jperio,
                      opts={"nvor_scheme": abi.VOR_NAMES[scheme], "nn_een_e3f": jpk % 2})
    rng = np.random.default_rng(jpk)
    if not uniform:
        for n in ("e3t_n", "e3u_n", "e3v_n"):
            d.arrays[n] *= 1.0 + 0.2 * rng.random(d.arrays[n].shape)
    hip.register(d)
    o, s3 = Oracle(d), (d.jpi, d.jpj, d.jpk)
    un, vn, wn, ua, va = (np.asfortranarray(rng.standard_normal(s3)) for _ in range(5))
    g = [dev(a) for a in (un, vn, wn, ua, va)]
    o.dyn_vor(1, un, vn, ua, va)
    hip.dyn_vor(1, g[0], g[1], g[3], g[4])
    o.dyn_adv(1, un, vn, wn, ua, va)
    hip.dyn_adv(1, *g)
    sync(hip)
    for n, w, x in zip(("ua", "va"), (ua, va), g[3:]):
        check(host(x, s3), w, what=f"{jpi}x{jpj}x{jpk} jperio {jperio} {scheme} {n}")
