"""Passes over few lines: tiles are halved until a pass has 192 of them or its
rows are 64 bytes.  Sizes on both sides of that line, odd tile heights, and
fewer lines than the least tile holds.  Oracle and tolerances of
test_gpu_fft.py: 1e-12 / 1e-6 relative L2 against the FP64 DFT."""
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
    (1, (3, 3, 1575), (1, 1, 1)),      # nine lines of the long axis
    (12, (61, 21, 50), (2, 3, 2)),     # a direct-sum prime, uneven ranks
    (4, (24, 1575), (2, 2)),
    (1, (64, 32, 48), (1, 1, 1)),      # tiles of both sides of 192 by pass and type
    (6, (75, 200), (6, 1)),
])
def test_small_tiles(C, P, shape, grid, dbl):
    fwd, rt, _ = run_split(C, P, shape, grid, slab=0, dbl=dbl)
    tol = TOL64 if dbl else TOL32
    assert fwd < tol and rt < tol, (fwd, rt)
