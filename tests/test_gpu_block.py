"""Block passes (several whole axes in one tile) at the edges of their rule:
whole arrays, planes with a ragged line tail, mixed radices, tile capacity
and one beyond it, stage groups of the phase order.  Oracle and tolerances
of test_gpu_fft.py: 1e-12 / 1e-6 relative L2 against the FP64 DFT."""
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


def check(C, P, shape, grid, dbl, **kw):
    fwd, rt, _ = run_split(C, P, shape, grid, dbl=dbl, **kw)
    tol = TOL64 if dbl else TOL32
    assert fwd < tol and rt < tol, (fwd, rt)


@pytest.mark.parametrize("dbl", [True, False])
@pytest.mark.parametrize("shape,grid,P", [
    ((2, 2), (1, 2), 2),            # the smallest: two radix-2 stages
    ((16, 16, 16), (1, 2, 2), 4),   # 4096 points: one tile of complex doubles
    ((16, 32, 16), (2, 2, 1), 4),   # 8192: one tile of complex floats, planes of doubles
    ((15, 14, 12), (1, 1, 1), 1),   # radices 3, 5, 7: nothing fused at either end
    ((7, 9, 8), (1, 1, 1), 1),
    ((64, 64, 64), (1, 2, 2), 4),   # planes, then lines of the first axis
    ((50, 64, 64), (5, 1, 1), 5),   # lines of 50 points
    ((45, 30, 42), (1, 1, 1), 1),   # planes of 1260 with a tail of lines
    ((11, 40, 48), (1, 1, 1), 1),   # the line axis has a prime without a block radix
    ((3, 4, 5, 6), (1, 2, 1, 2), 4),  # four axes: no block pass
    ((2048, 2), (1, 1), 1),         # a long row beside a short axis
    ((2, 4096), (1, 1), 1),         # beyond a tile of doubles, one tile of floats
])
def test_small_arrays(C, shape, grid, P, dbl):
    check(C, P, shape, grid, dbl, B=[1] * (len(shape) - 1) + [shape[-1]])
    check(C, P, shape, grid, dbl, slab=0)


@pytest.mark.parametrize("dbl,plain", [(True, False), (False, False), (False, True)])
@pytest.mark.parametrize("shape,grid,P,B", [
    ((64, 64, 64), (1, 2, 2), 4, [8, 8, 8]),        # 8 x 8 x 8 in both stages
    ((32, 64, 96), (2, 2, 2), 8, [2, 4, 6]),        # mixed radices, groups of three
    ((64, 128, 128), (1, 2, 2), 4, [4, 32, 32]),    # two axes and one
    ((40, 60, 36), (1, 2, 2), 4, [4, 6, 6]),        # uneven ranks: line passes
    ((26, 32, 64), (1, 2, 2), 4, [13, 4, 8]),       # a prime without a block radix
])
def test_phase_order_stages(C, shape, grid, P, B, dbl, plain):
    check(C, P, shape, grid, dbl, B=B, phased=True, plain_twiddles=plain)
