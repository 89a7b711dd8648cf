"""Ranks with strides of their own (uneven packed blocks): the FFT pass's
per-line addressing at its limits, and the dense intermediates of the fused
program when blocks are uneven or a second axis has to be split.  Oracle and
tolerances of test_gpu_fft.py: 1e-12 / 1e-6 relative L2 against the FP64 DFT."""
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


@pytest.mark.parametrize("dbl", [True, False])
@pytest.mark.parametrize("P,shape,grid", [
    (6, (30, 42, 20), (1, 2, 3)),     # uneven blocks of the slowest axis
    (12, (50, 2, 3), (4, 1, 3)),      # slow axes too short: two axes in blocks
    (8, (2, 3, 70), (1, 1, 8)),       # many positions along the first pass's axis
    (6, (33, 50), (3, 2)),            # 2D: the intermediate's slow axis is the pass's own
    (5, (17, 26, 9), (5, 1, 1)),      # direct-sum prime with uneven ranks
])
def test_uneven_ranks(C, P, shape, grid, dbl):
    fwd, rt, _ = run_split(C, P, shape, grid, slab=0, dbl=dbl)
    tol = TOL64 if dbl else TOL32
    assert fwd < tol and rt < tol, (fwd, rt)


@pytest.mark.parametrize("dbl", [True, False])
@pytest.mark.parametrize("n1,ranks", [
    (129, 8),       # a short last block: a table row per point
    (2101, 700),    # positions x lines at the LDS limit
    (2101, 1100),   # more positions than LDS holds: the line table in memory
])
def test_line_positions(C, n1, ranks, dbl):
    shape = (3, n1, 4)
    comm = C.dm_world_create(ranks)
    inp = C.makePackedDecomp(comm, 3, dm.ptrs([C.makeLocalDecomp(3), C.makeBlockDecomp(n1, ranks), C.makeLocalDecomp(4)]))
    out = C.makePackedDecomp(comm, 3, dm.ptrs([C.makeLocalDecomp(n) for n in shape]))
    ct = np.complex128 if dbl else np.complex64
    es = np.dtype(ct).itemsize
    per = 12 * (-(-n1 // ranks))
    a, b = dm.DistBuffer(comm, per * es), dm.DistBuffer(comm, 12 * n1 * es)
    rng = np.random.default_rng(n1 + ranks)
    x = (rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)).astype(ct)
    bs = -(-n1 // ranks)
    for r in range(-(-n1 // bs)):
        a.put(r, x[:, r * bs:(r + 1) * bs])
    p = C.dm_plan_axis_fft(inp, out, 1, 1 if dbl else 0, dm.FFTW_FORWARD)
    assert p and C.dm_run_axis_fft(p, a.ptr, b.ptr) == 0
    want = np.fft.fft(x.astype(np.complex128), axis=1)
    tol = TOL64 if dbl else TOL32
    assert rel_l2(b.get(0, 12 * n1 * es, ct).astype(np.complex128), want.ravel()) < tol
    q = C.dm_plan_axis_fft(out, inp, 1, 1 if dbl else 0, dm.FFTW_FORWARD)
    b.put(0, x)
    assert q and C.dm_run_axis_fft(q, b.ptr, a.ptr) == 0
    got = np.concatenate([a.get(r, x[:, r * bs:(r + 1) * bs].nbytes, ct).reshape(3, -1, 4)
                          for r in range(-(-n1 // bs))], axis=1)
    assert rel_l2(got.astype(np.complex128), want) < tol
    for f in (p, q):
        C.dm_free_axis_fft(f)
    a.free()
    b.free()
    for d in (inp, out):
        C.freeDecomp(d)
    C.dm_world_free(comm)
