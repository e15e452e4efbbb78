"""tra_adv_fct_coef_tl and tra_nxt_one against the calls they stand for: the
same operations, so the same bits (level counts around the blocks of levels,
closed and cyclic sides)."""
import numpy as np
import pytest

from nemo_hip import configs
from oracle.oracle import Oracle
from test_gpu_parity import dev, sync

torch = pytest.importorskip("torch")


@pytest.mark.gpu
@pytest.mark.parametrize("kn", [(2, 2), (4, 4)])
@pytest.mark.parametrize("jpi,jpj,jpk,jperio", [(33, 27, 5, 0), (34, 26, 6, 1), (70, 31, 33, 7)])
def test_fused_calls_equal_the_separate_ones(hip, jpi, jpj, jpk, jperio, kn):
    d = configs.basin(jpi, jpj, jpk, seed=jpk, jperio=jperio)
    hip.register(d)
    o, S = Oracle(d), configs.make_state(d, seed=6)
    s3 = (d.jpi, d.jpj, d.jpk)
    z = [np.zeros(s3, order="F") for _ in range(3)]
    o.tra_adv_trp(S["un"], S["vn"], S["wn"], *z)
    trp, (tb, tn, a0) = [dev(a) for a in z], [dev(S[n][..., 0]) for n in ("tsb", "tsn", "tsa")]
    p2dt = 2.0 * d.opts["rdt"]
    c0, c1 = ([torch.zeros_like(tb) for _ in range(3)] for _ in range(2))
    t0, t1 = a0.clone(), a0.clone()
    torch.cuda.synchronize()
    hip.tra_adv_fct_coef(p2dt, *trp, tb, tn, *c0, kn=kn)
    hip.tra_adv_fct_tl(p2dt, *trp, tb, tn, *c0, t0, kn=kn)
    hip.tra_adv_fct_coef_tl(p2dt, *trp, tb, tn, *c1, t1, kn=kn)
    sync(hip)
    for x, y in zip(c0 + [t0], c1 + [t1]):
        assert torch.equal(x, y)
    for kt in (1, 5):
        two = [torch.cat([x, x]) for x in (tb, tn, t0)]
        one = [x.clone() for x in (tb, tn, t0)]
        torch.cuda.synchronize()
        hip.tra_nxt(kt, *two)
        hip.tra_nxt_one(kt, *one)
        sync(hip)
        for x, y in zip(two, one):
            assert torch.equal(x[:y.numel()], y)
