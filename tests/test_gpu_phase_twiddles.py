"""The phase order's twiddles where the first rank's own factors are all 1
(it holds only the first coordinate of every split axis): the other ranks'
are not.  Oracle and tolerances of test_gpu_fft.py."""
import pytest

import decomp_mpi_amd as dm
from test_gpu_fft import TOL32, TOL64, run_split

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def C():
    C = dm.lib()
    if not C.dm_device_available():
        pytest.skip("no HIP device")
    return C


@pytest.mark.parametrize("dbl", [True, False])
@pytest.mark.parametrize("P,shape,grid", [
    (32, (13, 40, 32), (1, 4, 8)),
    (32, (8, 16, 15), (2, 4, 4)),
    (2, (4, 3, 5), (2, 1, 1)),      # one split axis, 2 x 2
])
def test_first_rank_without_factors(C, P, shape, grid, dbl):
    fwd, rt, _ = run_split(C, P, shape, grid, slab=0, dbl=dbl, phased=True)
    tol = TOL64 if dbl else TOL32
    assert fwd < tol and rt < tol, (fwd, rt)
