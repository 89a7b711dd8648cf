"""Plane tiles whose columns take three power-of-two stages (128 and 256
points in butterflies of up to 8), alone and with odd radices, and rows of as
many.  Tolerances of test_gpu_fft.py against numpy's FP64 DFT."""
import ctypes

import numpy as np
import pytest

import decomp_mpi_amd as dm
from test_gpu_fft import TOL32, TOL64

pytestmark = pytest.mark.gpu

SHAPES = [(3, 128, 32), (2, 256, 16), (5, 256, 3), (2, 128, 30), (2, 192, 20), (3, 15, 256), (2, 32, 128), (1, 256, 1)]


@pytest.fixture(scope="module")
def C():
    C = dm.lib()
    if not C.dm_device_available():
        pytest.skip("no HIP device")
    return C


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("direction", [-1, 1])
@pytest.mark.parametrize("dbl", [0, 1])
def test_long_columns(C, dbl, direction, order):
    comm = C.dm_world_create(1)
    ct = np.complex128 if dbl else np.complex64
    es = np.dtype(ct).itemsize
    offs = np.concatenate([[0], np.cumsum([-(-int(np.prod(s)) // 32) * 32 for s in SHAPES])])
    buf = dm.DistBuffer(comm, int(offs[-1]) * es)
    rng = np.random.default_rng(7)
    xs = [(rng.uniform(-1, 1, s) + 1j * rng.uniform(-1, 1, s)).astype(ct) for s in SHAPES]
    plan = C.dm_batch_plan(len(SHAPES), 3, dm.ints([n for s in SHAPES for n in s]), dbl, direction)
    ptrs = (ctypes.c_void_p * len(SHAPES))(*[buf.ptr + int(o) * es for o in offs[:-1]])
    assert plan and C.dm_batch_bind(plan, ptrs) == 0
    assert C.dm_batch_set_schedule(plan, dm.DM_BATCH_TILE_PLANES, order) == 0
    for x, o in zip(xs, offs):
        buf.put(0, x, int(o) * es)
    assert C.dm_batch_run(plan, C.dm_get_stream(comm)) == 0
    C.dm_synchronize(comm)
    for x, o, s in zip(xs, offs, SHAPES):
        got = buf.get(0, x.nbytes, ct, int(o) * es).reshape(s).astype(np.complex128)
        x64 = x.astype(np.complex128)
        want = np.fft.fftn(x64) if direction == -1 else np.fft.ifftn(x64) * x64.size
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        assert err < (TOL64 if dbl else TOL32), (s, err)
    C.dm_batch_free(plan)
    buf.free()
    C.dm_world_free(comm)
