"""The reshape's tile, row and general kernels at the edges of their tiles:
every element size, both walks (transposed and shared fastest axis), even
and uneven ranks, narrow tile axes, batch tails, buffers beyond 4 GiB.
Bit-exact against the oracle on every destination byte."""
import ctypes

import numpy as np
import pytest

import decomp_mpi_amd as dm
import oracle
from helpers import make_pair

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def C():
    C = dm.lib()
    if not C.dm_device_available():
        pytest.skip("no HIP device")
    return C


def reshape(C, P, src, dst, elem, src_strides=None, dst_strides=None, slot=0):
    """src / dst: descriptors; slot: bytes per rank of both buffers (0: what
    the larger block needs)."""
    comm = C.dm_world_create(P)
    ps, os_ = make_pair(C, comm, P, src, None, src_strides)
    pd, od = make_pair(C, comm, P, dst, None, dst_strides)
    t = ctypes.c_void_p()
    C.dm_type_contiguous(elem, dm.mpi_type("byte"), ctypes.byref(t))
    plan = C.makeReshapePlan(comm, t, ps, pd)
    assert plan
    sn, dn = int(max(os_.extents)) * elem, int(max(od.extents)) * elem
    sb, db = dm.DistBuffer(comm, max(sn, slot)), dm.DistBuffer(comm, max(dn, slot))
    rng = np.random.default_rng(elem + P)
    hs = rng.integers(0, 256, (P, sn), dtype=np.uint8)
    hd = rng.integers(0, 256, (P, dn), dtype=np.uint8)
    sb.put_all(hs)
    db.put_all(hd)
    C.runReshapePlan(comm, plan, sb.ptr, db.ptr)
    got = db.get_all(dn, np.uint8)
    want = hd.copy()
    oracle.reshape(os_, od, hs, want, elem)
    C.freeReshapePlan(plan)
    for b in (sb, db):
        b.free()
    for d in (ps, pd):
        C.freeDecomp(d)
    C.dm_world_free(comm)
    assert np.array_equal(got, want)


SIZES = [1, 2, 4, 8, 12, 16, 20, 24, 48]
BLOCK = [("block", 5, 1), ("block", 67, 2), ("block", 130, 2)]


@pytest.mark.parametrize("elem", SIZES)
@pytest.mark.parametrize("dst,strides", [
    # transposed, even strides: 65 and 130 wide tile axes
    ([("block", 5, 1), ("rotate", 9, ("block", 67, 1)), ("block", 130, 4)], [67 * 33, 1, 67]),
    # transposed over a narrow axis (5), batch tail
    ([("local", 5), ("block", 67, 2), ("block", 130, 2)], [1, 5 * 65, 5]),
    # shared fastest axis: rows of 33 and of 130
    ([("block", 5, 1), ("block", 67, 1), ("block", 130, 4)], None),
    ([("block", 5, 2), ("rotate", 30, ("block", 67, 2)), ("local", 130)], None),
    # the first axis interleaved, the shared one rotated
    ([("block", 5, 5), ("local", 67), ("rotate", 1, ("local", 130))], None),
])
def test_walks(C, elem, dst, strides):
    reshape(C, 5, BLOCK, dst, elem, None, strides)


@pytest.mark.parametrize("elem", SIZES)
def test_rows_only(C, elem):
    """One axis, and long rows with too few neighbours for the row kernel."""
    reshape(C, 3, [("block", 2500, 3)], [("rotate", 700, ("block", 2500, 2))], elem)
    reshape(C, 3, [("block", 2, 1), ("block", 2500, 3)], [("block", 2, 2), ("rotate", 7, ("local", 2500))], elem)


@pytest.mark.parametrize("elem", [4, 12, 16])
def test_partly_owned(C, elem):
    """Coordinates that sit on ranks the decomposition does not use stay
    where they are (the general kernels)."""
    reshape(C, 6, [("single", 40, 0, 1), ("block", 50, 3)], [("block", 40, 2), ("block", 50, 3)], elem)


@pytest.mark.parametrize("elem", [8, 12])
def test_many_positions(C, elem):
    """More (a, b) position pairs of uneven ranks than a workgroup's table."""
    src = [("block", 45, 23), ("block", 47, 24)]
    reshape(C, 23 * 24, src, [("rotate", 3, ("local", 45)), ("block", 47, 500)], elem, None, [1, 45])


@pytest.mark.parametrize("elem", [4, 24])
@pytest.mark.parametrize("dst,strides", [
    ([("block", 6, 2), ("local", 70), ("local", 70)], [70 * 70, 1, 70]),
    ([("block", 6, 1), ("block", 70, 2), ("local", 70)], None),
])
def test_beyond_4gib(C, elem, dst, strides):
    reshape(C, 2, [("block", 6, 1), ("block", 70, 1), ("block", 70, 2)], dst, elem, None, strides, slot=(9 << 28) + 48)
