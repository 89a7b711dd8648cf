"""Split transforms whose start layout leaves gaps between its rows and
elements, and whose output is a layout of the caller's (dm_split_set_output,
with its axes in another order): block passes, planes and lines, long axes in
two passes.  The gaps keep what they held.  Against numpy's FP64 DFT with the
tolerances of test_gpu_fft.py."""
import numpy as np
import pytest

import decomp_mpi_amd as dm
from helpers import make_pair, rel_l2
from test_gpu_fft import TOL32, TOL64, block_start, owned_mask, placement
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def C():
    C = dm.lib()
    if not C.dm_device_available():
        pytest.skip("no HIP device")
    return C


def gapped(shape, grid, order, step, pad):
    """Memory strides with the axes in `order` (fastest first), elements
    `step` apart and every further axis `pad` longer than it has to be."""
    strides, at = [0] * len(shape), step
    for d in order:
        strides[d] = at
        at *= -(-shape[d] // grid[d]) + pad
    return strides


@pytest.mark.parametrize("dbl", [True, False])
@pytest.mark.parametrize("step,pad", [(1, 1), (3, 0)])
@pytest.mark.parametrize("permute", [False, True])
@pytest.mark.parametrize("shape,grid", [
    ((16, 16, 16), (1, 2, 2)),     # one block pass
    ((64, 32, 64), (1, 2, 2)),     # planes, then lines
    ((30, 42, 50), (1, 2, 3)),     # lines
    ((2048, 1040), (4, 1)),        # a long axis in two passes
    ((24, 2048, 64), (2, 2, 1)),
])
def test_gaps_and_chosen_output(C, shape, grid, permute, step, pad, dbl):
    nd, P = len(shape), int(np.prod(grid))
    comm = C.dm_world_create(P)
    ct, es = (np.complex128, 16) if dbl else (np.complex64, 8)
    descs = block_start(shape, grid)
    order = list(range(nd))[::-1] if not permute else list(range(1, nd)) + [0]
    ps, os_ = make_pair(C, comm, P, descs, None, gapped(shape, grid, order, step, pad))
    per = int(max(os_.extents))
    length = 4 * max(per, int(np.prod(shape)) // P + 1) + 64
    dat, work = dm.DistBuffer(comm, per * es), dm.DistBuffer(comm, length * es)
    plan = (C.makeSplitPlan if dbl else C.makeSplitPlanf)(0, ps, dat.ptr, length, work.ptr)
    assert plan
    sp = dm.split_plan(plan)
    A = [sp.A_factors[i] for i in range(nd)]
    B = [n // a for n, a in zip(shape, A)]
    rng = np.random.default_rng(nd + step)
    x = (rng.uniform(-1, 1, (P, per)) + 1j * rng.uniform(-1, 1, (P, per))).astype(ct)
    glob = x[placement(os_)].astype(np.complex128)
    want = np.fft.fftn(glob)
    tol = TOL64 if dbl else TOL32
    pos = np.meshgrid(*[np.arange(n) // b + a * (np.arange(n) % b) for n, a, b in zip(shape, A, B)], indexing="ij")
    flipped = oracle.split_decomps(P, A, B, oracle.processor_grid(P, A), oracle.processor_grid(P, B))
    flipped = flipped[1 if any(a > 1 for a in A) else 0]
    own = None
    for chosen in (False, True):
        if chosen:  # the same blocks, the first axis fastest
            own = make_pair(C, comm, P, descs, None, gapped(shape, grid, range(nd), 1, 0))
            if int(max(own[1].extents)) > sp.extent:
                break
            assert C.dm_split_set_output(plan, own[0]) == 0
        dat.put_all(x)
        C.runSplitPlan(plan, dm.FFTW_FORWARD)
        got = work.get_all(sp.extent * es, ct)
        if chosen:
            spec = got[placement(own[1])]
        else:
            rank, off = placement(flipped)
            spec = got[rank[tuple(pos)], off[tuple(pos)]]
        assert rel_l2(spec.astype(np.complex128), want) < tol
        dat.put_all(-x)  # (a value of its own in the gaps)
        C.runSplitPlan(plan, dm.FFTW_BACKWARD)
        back = dat.get_all(per * es, ct)
        mask = owned_mask(os_, per)
        assert rel_l2(back[mask].astype(np.complex128) / glob.size, x[mask].astype(np.complex128)) < tol
        assert np.array_equal(back[~mask], -x[~mask])
    C.freeSplitPlan(plan)
    for b in (dat, work):
        b.free()
    for d in [ps] + ([own[0]] if own else []):
        C.freeDecomp(d)
    C.dm_world_free(comm)
