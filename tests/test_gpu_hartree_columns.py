"""The z passes of the Hartree potential at the edge of their two forms (16 and 8 columns per block, or 4 where few
columns have many planes: at least 64 planes of at most 4096 points), column counts that do not fill a block,
one and two spin channels, against the CPU oracle.

Tolerance 1e-12 relative as for the other potential calls: sums of at most 256 terms per pass, five passes."""
import pytest

from tests import test_gpu_hartree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(5, 7, 63), (5, 7, 64), (13, 5, 65), (6, 9, 129), (7, 5, 255), (64, 64, 64), (64, 65, 64)])
@pytest.mark.parametrize("nspin", [1, 2])
def test_z_pass_columns(oracle_lib, n, nspin):
    test_gpu_hartree.test_hartree_extents(oracle_lib, n, nspin)
