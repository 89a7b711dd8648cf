"""Axes too long for wide rows in one pass: two passes with a twiddle between
them, at the lengths where the rule starts, with mixed radices, several long
axes, layouts that do not separate (which keep the one-pass form), and
ranks.  Oracle and tolerances of test_gpu_fft.py."""
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
@pytest.mark.parametrize("shape,grid,P,desc", [
    ((1024, 1056), (1, 1), 1, None),        # the last length in one pass
    ((2048, 1050), (4, 1), 4, None),        # 32 x 64 points, a ragged tail of lines
    ((4096, 520), (2, 2), 4, None),         # 64 x 64
    ((2160, 1000), (1, 2), 2, None),        # 45 x 48: odd first radices, one pass
    ((2400, 900), (3, 2), 6, None),         # 48 x 50
    ((2187, 960), (1, 1), 1, None),         # 27 x 81: one pass
    ((512, 4096), (2, 2), 4, None),         # the long axis is the contiguous one
    ((2048, 2048), (2, 4), 8, None),
    ((4096, 6, 100), (2, 1, 2), 4, None),   # 3D, long axis slowest
    ((6, 4096, 90), (2, 2, 1), 4, None),    # in the middle
    ((2048, 1, 1100), (4, 1, 1), 4, None),
    ((2048, 1024), (4, 1), 4, [("rotate", 100, ("block", 2048, 4)), ("block", 1024, 1)]),  # does not separate
    ((64, 4096), (1, 1), 1, None),          # below the size where it pays
])
def test_long_axes(C, shape, grid, P, desc, dbl):
    fwd, rt, _ = run_split(C, P, shape, grid, slab=0, dbl=dbl, start_descs=desc)
    tol = TOL64 if dbl else TOL32
    assert fwd < tol and rt < tol, (fwd, rt)
