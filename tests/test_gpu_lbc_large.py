"""lbc_lnk over more than 4 GiB, where a 32-bit byte offset from the array's
first element would wrap to its first levels: the FCT fills the ring of up to
four arrays of a domain in one launch, and only one of them is sure to stay
below 4 GiB.  The fill copies and clears, so the result is exact."""
import pytest

from nemo_hip import configs

torch = pytest.importorskip("torch")


@pytest.mark.gpu
@pytest.mark.parametrize("jperio", [0, 1, 2])
def test_ring_of_levels_beyond_4_gib(hip, jperio):
    d = configs.gyre_like(1024, 1024, 3, jperio=jperio)
    hip.register(d)
    nk = (1 << 32) // (d.jpi * d.jpj * 8) + 3          # the last three levels lie beyond 4 GiB
    a = torch.rand((nk, d.jpj, d.jpi), dtype=torch.float64, device="cuda")
    w = a.clone()
    if jperio == 1:
        w[:, :, 0], w[:, :, -1] = w[:, :, -2].clone(), w[:, :, 1].clone()
    else:
        w[:, :, 0] = w[:, :, -1] = 0.5
    if jperio == 2:
        w[:, 0], w[:, -1] = w[:, -2].clone(), w[:, 1].clone()
    else:
        w[:, 0] = w[:, -1] = 0.5
    torch.cuda.synchronize()
    hip.lbc_lnk(a, nk, "T", pval=0.5)
    hip.sync()
    assert torch.equal(a, w)
