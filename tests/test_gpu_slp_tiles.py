"""ldf_slp where its tiles change their shape: cyclic directions of one tile,
two, and more (the first and the last tile carry the wider halo of the seam),
one point short of the next number of tiles and one beyond, with one to four
and more levels per workgroup.  Against the oracle with the parity tests'
1e-12."""
import pytest

from test_gpu_slp_regions import test_slopes_and_viscosity_at_region_edges as check_slopes

# interior points at the edges: 24, 25, 52, 53, 80, 81 along i; 8, 9, 20, 21, 32, 33 along j
SIZES = [(26, 10, 6, 7), (27, 11, 31, 7), (54, 22, 12, 7), (55, 23, 31, 7), (56, 24, 40, 7), (82, 34, 9, 7), (83, 35, 20, 7),
         (111, 60, 12, 7), (27, 40, 20, 1), (55, 31, 31, 1), (83, 50, 6, 1), (40, 11, 20, 2), (33, 23, 31, 2), (60, 35, 40, 2)]


@pytest.mark.gpu
@pytest.mark.parametrize("jpi,jpj,jpk,jperio", SIZES)
def test_tiles_of_cyclic_directions(hip, jpi, jpj, jpk, jperio):
    check_slopes(hip, jpi, jpj, jpk, jperio)
