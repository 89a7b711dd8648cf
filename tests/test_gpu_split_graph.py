"""A split plan that has run in one direction is ready for a graph of the
other: nothing is allocated or copied then.  Every replay against the eager
result, bit for bit."""
import ctypes

import numpy as np
import pytest

import decomp_mpi_amd as dm
from helpers import make_pair
from test_gpu_fft import block_start

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def C():
    C = dm.lib()
    if not C.dm_device_available():
        pytest.skip("no HIP device")
    return C


class Hip:
    """The HIP runtime that the library itself is bound to."""

    def __init__(self):
        self.lib = ctypes.CDLL(dm.LIB_PATH)  # (its dependencies' symbols with it)

    def call(self, name, *args):
        rc = getattr(self.lib, name)(*args)
        assert rc == 0, (name, rc)

    def stream(self):
        s = ctypes.c_void_p()
        self.call("hipStreamCreateWithFlags", ctypes.byref(s), 1)
        return s

    def record(self, stream, work):
        """work() recorded from `stream` into an executable graph."""
        graph, run = ctypes.c_void_p(), ctypes.c_void_p()
        self.call("hipStreamBeginCapture", stream, 0)
        work()
        self.call("hipStreamEndCapture", stream, ctypes.byref(graph))
        self.call("hipGraphInstantiate", ctypes.byref(run), graph, None, None, ctypes.c_size_t(0))
        self.call("hipGraphDestroy", graph)
        return run


@pytest.mark.parametrize("first", ["forward", "backward"])
@pytest.mark.parametrize("shape,grid", [
    ((16, 16, 16), (1, 2, 2)),       # one block pass
    ((60, 90, 84), (1, 2, 2)),       # line passes
    ((2048, 1100), (2, 2)),          # a long axis in two passes
])
def test_other_direction_in_a_graph(C, shape, grid, first):
    P, N = int(np.prod(grid)), int(np.prod(shape))
    ahead, other = (dm.FFTW_FORWARD, dm.FFTW_BACKWARD) if first == "forward" else (dm.FFTW_BACKWARD, dm.FFTW_FORWARD)
    hip = Hip()
    stream = hip.stream()
    rng = np.random.default_rng(N)

    def plan_of():
        comm = C.dm_world_create(P)
        assert C.dm_set_stream(comm, stream) == 0 and C.dm_set_async(comm, 1) == 0
        ps, os_ = make_pair(C, comm, P, block_start(shape, grid))
        per = int(max(os_.extents))
        length = 4 * max(per, N // P + 1)
        dat, work = dm.DistBuffer(comm, per * 16), dm.DistBuffer(comm, length * 16)
        plan = C.makeSplitPlan(0, ps, dat.ptr, length, work.ptr)
        assert plan
        return comm, plan, dat, work, per, length

    def fill(dat, work, per, length, d, w):
        hip.call("hipStreamSynchronize", stream)
        dat.put_all(d)
        work.put_all(w)

    def result(dat, work, per, plan):
        hip.call("hipStreamSynchronize", stream)
        if other == dm.FFTW_BACKWARD:
            return dat.get_all(per * 16, np.complex128).copy()
        return work.get_all(dm.split_plan(plan).extent * 16, np.complex128).copy()

    made = [plan_of(), plan_of()]
    _, _, _, _, per, length = made[0]
    d = rng.uniform(-1, 1, (P, per)) + 1j * rng.uniform(-1, 1, (P, per))
    w = rng.uniform(-1, 1, (P, length)) + 1j * rng.uniform(-1, 1, (P, length))
    # eager, on a plan of its own
    comm, plan, dat, work, _, _ = made[0]
    fill(dat, work, per, length, d, w)
    C.runSplitPlan(plan, other)
    want = result(dat, work, per, plan)
    # recorded after one run in the other direction only
    comm, plan, dat, work, _, _ = made[1]
    fill(dat, work, per, length, d, w)
    C.runSplitPlan(plan, ahead)
    hip.call("hipStreamSynchronize", stream)
    graph = hip.record(stream, lambda: C.runSplitPlan(plan, other))
    for k in range(3):
        fill(dat, work, per, length, d, w)
        hip.call("hipGraphLaunch", graph, stream)
        got = result(dat, work, per, plan)
        # (slots past a rank's own points hold what the buffers held)
        assert np.array_equal(got, want), k
    hip.call("hipGraphExecDestroy", graph)
    for comm, plan, dat, work, _, _ in made:
        C.freeSplitPlan(plan)
        dat.free()
        work.free()
        C.dm_world_free(comm)
    hip.call("hipStreamDestroy", stream)
