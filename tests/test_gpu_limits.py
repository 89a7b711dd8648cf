"""Calls at the limits of a workgroup's LDS and of a plan's tables.  Oracle
and tolerances of test_gpu_fft.py: 1e-12 / 1e-6 relative L2 against the FP64
DFT."""
import itertools

import numpy as np
import pytest

import decomp_mpi_amd as dm
from helpers import rel_l2
from test_gpu_fft import TOL32, TOL64, run_split

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def C():
    C = dm.lib()
    if not C.dm_device_available():
        pytest.skip("no HIP device")
    return C


class Blocks:
    """Packed blocks of shape over grid: the decomposition, and its slots."""

    def __init__(self, C, comm, shape, grid):
        self.C = C
        self.sizes = [-(-n // g) for n, g in zip(shape, grid)]
        self.decomp = C.makePackedDecomp(comm, len(shape), dm.ptrs([C.makeBlockDecomp(n, g) for n, g in zip(shape, grid)]))
        self.parts = [tuple(slice(q * s, min(n, (q + 1) * s)) for q, s, n in zip(at, self.sizes, shape))
                      for at in itertools.product(*[range(g) for g in grid])]
        self.most = int(np.prod(self.sizes))

    def put(self, buf, x):
        for r, p in enumerate(self.parts):
            if x[p].size:
                buf.put(r, np.ascontiguousarray(x[p]))

    def get(self, buf, shape, ct):
        out = np.zeros(shape, ct)
        for r, p in enumerate(self.parts):
            n = out[p].size
            if n:
                out[p] = buf.get(r, n * np.dtype(ct).itemsize, ct).reshape(out[p].shape)
        return out


def axis_fft(C, shape, axis, gin, gout, dbl):
    """One axis transformed from blocks over gin into blocks over gout."""
    comm = C.dm_world_create(max(int(np.prod(gin)), int(np.prod(gout))))
    ct = np.complex128 if dbl else np.complex64
    es = np.dtype(ct).itemsize
    a, b = Blocks(C, comm, shape, gin), Blocks(C, comm, shape, gout)
    bi, bo = dm.DistBuffer(comm, a.most * es), dm.DistBuffer(comm, b.most * es)
    rng = np.random.default_rng(sum(shape))
    x = (rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)).astype(ct)
    a.put(bi, x)
    p = C.dm_plan_axis_fft(a.decomp, b.decomp, axis, 1 if dbl else 0, dm.FFTW_FORWARD)
    assert p and C.dm_run_axis_fft(p, bi.ptr, bo.ptr) == 0
    err = rel_l2(b.get(bo, shape, ct).astype(np.complex128), np.fft.fft(x.astype(np.complex128), axis=axis))
    C.dm_free_axis_fft(p)
    for buf in (bi, bo):
        buf.free()
    for d in (a.decomp, b.decomp):
        C.freeDecomp(d)
    C.dm_world_free(comm)
    assert err < (TOL64 if dbl else TOL32), err


@pytest.mark.parametrize("dbl", [True, False])
@pytest.mark.parametrize("shape,gin,gout", [
    ((512, 65, 130), (32, 2, 1), (32, 2, 1)),   # the wide tile and two sides' line data: 160.25 KiB
    ((512, 65, 130), (1, 2, 1), (64, 2, 1)),    # one side's
    ((1024, 65, 70), (64, 2, 1), (64, 2, 1)),
])
def test_line_data_beside_wide_tile(C, shape, gin, gout, dbl):
    axis_fft(C, shape, 0, gin, gout, dbl)


@pytest.mark.parametrize("dbl", [True, False])
def test_more_positions_than_lds_on_both_sides(C, dbl):
    axis_fft(C, (6, 2101, 5), 1, (1, 1100, 1), (1, 1100, 1), dbl)


@pytest.mark.parametrize("dbl", [True, False])
@pytest.mark.parametrize("shape,axis,gin,gout", [
    ((5, 50, 33), 1, (2, 6, 1), (2, 6, 1)),     # the most positions that are kept
    ((5, 50, 33), 1, (2, 7, 1), (2, 3, 1)),     # one more on one side
    ((5, 50, 33), 1, (1, 6, 1), (1, 10, 1)),    # and on the other
    ((9, 300, 8), 1, (2, 7, 1), (2, 100, 1)),
    ((7, 5, 61), 2, (2, 1, 20), (2, 1, 20)),    # a direct-sum prime, contiguous axis
    ((385, 65, 66), 0, (12, 2, 1), (12, 2, 1)), # the wide tile
])
def test_kept_positions_and_beyond(C, shape, axis, gin, gout, dbl):
    axis_fft(C, shape, axis, gin, gout, dbl)


@pytest.mark.parametrize("dbl", [True, False])
@pytest.mark.parametrize("P,shape,grid", [
    (4, (33, 1024), (2, 2)),       # the longest line of 64-byte rows
    (4, (33, 1050), (2, 2)),       # one beyond, and blocks of 33 are uneven
    (12, (26, 3025), (6, 2)),
    (6, (1050, 35), (3, 2)),       # the long axis last: dense all the same
    (6, (5, 1100, 14), (1, 3, 2)),
])
def test_uneven_intermediates_of_long_lines(C, P, shape, grid, dbl):
    fwd, rt, _ = run_split(C, P, shape, grid, slab=0, dbl=dbl)
    tol = TOL64 if dbl else TOL32
    assert fwd < tol and rt < tol, (fwd, rt)


@pytest.mark.parametrize("dbl", [True, False])
@pytest.mark.parametrize("shape,axis,gin,gout", [
    ((32, 39), 0, (2, 1), (1, 3)),   # complex double: the most points that are not spread over workgroups
    ((40, 32), 1, (3, 1), (1, 2)),   # and one line more
    ((79, 32), 1, (3, 1), (1, 2)),   # the same for complex float
    ((32, 80), 0, (2, 1), (1, 3)),
    ((104, 8), 0, (1, 1), (1, 1)),
    ((1, 2, 2), 1, (1, 1, 1), (1, 1, 1)),
    ((79, 45), 0, (2, 4), (2, 4)),   # a direct-sum prime: spread all the same
])
def test_passes_over_few_lines(C, shape, axis, gin, gout, dbl):
    axis_fft(C, shape, axis, gin, gout, dbl)
