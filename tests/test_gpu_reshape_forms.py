"""The reshape's tile forms at sizes where each is chosen: large tiles (64 MiB
a side and more) and narrow ones (a tile axis of at most 16 values, 128 MiB
over the element size and more), with remainders along both tile axes and the
batch, even and uneven ranks.  Bit-exact against the oracle on every
destination byte."""
import pytest

import decomp_mpi_amd as dm
from test_gpu_reshape_tiles import reshape

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def C():
    C = dm.lib()
    if not C.dm_device_available():
        pytest.skip("no HIP device")
    return C


def permuted(C, elem, shape, grid, mib):
    """Packed blocks (the last axis fastest) to blocks with the middle axis
    fastest; the first axis as long as `mib` MiB take."""
    n0 = mib * (1 << 20) // (elem * shape[0] * shape[1]) + 2
    n = (n0, *shape)
    src = [("block", a, g) for a, g in zip(n, grid)]
    most = [-(-a // g) for a, g in zip(n, grid)]
    P = grid[0] * grid[1] * grid[2]
    reshape(C, P, src, src, elem, dst_strides=[most[1] * most[2], 1, most[1]])


@pytest.mark.parametrize("elem", [1, 4, 8, 16])
@pytest.mark.parametrize("grid", [(1, 1, 2), (1, 2, 2)])  # even; uneven along the axis of 515
def test_large(C, elem, grid):
    permuted(C, elem, (515, 510), grid, 64)


@pytest.mark.parametrize("elem", [4, 8, 16])
@pytest.mark.parametrize("shape", [(13, 515), (515, 13), (16, 16)])
@pytest.mark.parametrize("grid", [(1, 1, 1), (2, 2, 3)])
def test_narrow(C, elem, shape, grid):
    permuted(C, elem, shape, grid, 128 // elem)
