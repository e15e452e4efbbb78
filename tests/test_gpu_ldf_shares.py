"""dyn_ldf_lap (and ldf_slp) where a workgroup takes several levels: shares of
two to sixteen levels with and without a remainder.  Against the oracle with the
parity tests' 1e-12."""
import pytest

from test_gpu_slp_regions import test_slopes_and_viscosity_at_region_edges as check_viscosity

SIZES = [(330, 100, 40, 0), (400, 120, 19, 1), (640, 200, 12, 0), (700, 420, 20, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("jpi,jpj,jpk,jperio", SIZES)
def test_shares_of_levels(hip, jpi, jpj, jpk, jperio):
    check_viscosity(hip, jpi, jpj, jpk, jperio)
