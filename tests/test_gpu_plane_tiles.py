"""Plane tiles of the batched FFT where their rule turns: several planes per
tile with a tail, the 256- and 512-thread classes, sides of one point, odd
sides, the largest side, both radix orders.  numpy's FP64 DFT; 1e-6 (complex
float) and 1e-12 (complex double) relative L2."""
import ctypes

import numpy as np
import pytest

import decomp_mpi_amd as dm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def C():
    C = dm.lib()
    if not C.dm_device_available():
        pytest.skip("no HIP device")
    return C


SHAPES = [(7, 16, 16), (5, 2, 2), (3, 1, 20), (3, 20, 1), (2, 1, 1), (3, 15, 21), (9, 48, 32), (2, 64, 64), (3, 96, 80),
          (2, 128, 64), (2, 256, 32), (2, 16, 256), (4, 26, 22), (1, 90, 91), (2, 12, 10)]


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("direction", [-1, 1])
@pytest.mark.parametrize("dbl", [0, 1])
def test_plane_tiles(C, dbl, direction, order):
    comm = C.dm_world_create(1)
    ct = np.complex128 if dbl else np.complex64
    es = np.dtype(ct).itemsize
    sizes = [int(np.prod(s)) for s in SHAPES]
    offs = np.concatenate([[0], np.cumsum([(n + 31) // 32 * 32 for n in sizes])])
    buf = dm.DistBuffer(comm, int(offs[-1]) * es)
    rng = np.random.default_rng(5)
    xs = [(rng.uniform(-1, 1, s) + 1j * rng.uniform(-1, 1, s)).astype(ct) for s in SHAPES]
    plan = C.dm_batch_plan(len(SHAPES), 3, dm.ints([v for s in SHAPES for v in s]), dbl, direction)
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
        assert err < (1e-12 if dbl else 1e-6), (s, err)
    C.dm_batch_free(plan)
    buf.free()
    C.dm_world_free(comm)
