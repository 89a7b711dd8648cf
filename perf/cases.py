"""The workloads whose speed this library is held to, through its public C ABI.

Each case is what a program that uses the library has it do: split 3D
transforms from tiny to 512^3, slab and pencil stages, reshapes between
decompositions, batches of uneven local transforms, and the request loop.

listed() names the fixed cases, draw(rng) makes further ones of the same
ranges, prepare(case, seed) builds inputs and plans, run(state) is one pass,
work(case) the bytes and operations a pass cannot do without, exact(case,
seed) the outputs in 64 bits from plain torch.
"""
import ctypes
import math
import random

import torch

import decomp_mpi_amd as dm
from decomp_mpi_amd import workloads

DEV = "cuda"
CDT = {"c128": torch.complex128, "c64": torch.complex64}


def listed():
    return [
        # The smallest split transform: a driver's first call on a 16^3 box,
        # four ranks, default (blocking) mode.  Launch and host latency.
        dict(name="split-16", kind="split", shape="16x16x16", grid="1x2x2", ranks=4, factors="", precision="c128",
             mode="forward", order="fused"),
        # A pencil code's three FFT stages with the reshapes between them,
        # 64^3 on a 2x2 grid.  Small launches back to back.
        dict(name="pencil-64", kind="pencil", shape="64x64x64", grid="2x2", ranks=4, precision="c128"),
        # Uneven blocks on six ranks, mixed radices: no layout is uniform.
        dict(name="split-ragged", kind="split", shape="90x126x100", grid="1x2x3", ranks=6, factors="",
             precision="c128", mode="forward", order="fused"),
        # Images / planes: the inverse of a long-axis 2D transform.
        dict(name="split-2d-back", kind="split", shape="4096x2048", grid="4x2", ranks=8, factors="",
             precision="c128", mode="backward", order="fused"),
        # The headline transform: 512^3 complex double from pencils on a 4x8
        # grid, with the split that the autotuner picks there.
        dict(name="split-512", kind="split", shape="512x512x512", grid="1x4x8", ranks=32, factors="1x64x1",
             precision="c128", mode="forward", order="fused"),
        # Its complex-float form, forward, scaled by 1/N, backward: one step
        # of a spectral solver.
        dict(name="split-512-c64-step", kind="split", shape="512x512x512", grid="1x4x8", ranks=32, factors="1x64x1",
             precision="c64", mode="step", order="fused"),
        # The reference's own phase order and default split (A = 16, B = 32):
        # what callers that read the phase timers run, and every transform
        # with an axis longer than one tile.
        dict(name="phases-512", kind="split", shape="512x512x512", grid="1x4x8", ranks=32, factors="",
             precision="c128", mode="forward", order="phases"),
        # The 512^3 int64 reshape chain: block -> rotated and permuted ->
        # interleaved on a 4x8 grid.
        dict(name="reshape-512", kind="chain", shape="512x512x512", ranks=32, shift="65x76x450"),
        # A field of 12-byte elements (three floats) from uneven blocks to
        # uneven rotated pencils on twelve ranks.
        dict(name="reshape-ragged", kind="reshape", shape="150x77x201", ranks=12, grid="2x3x2", dest="3x1x4",
             form="rotated", words=3),
        # 256 independent complex-float 3D transforms of uneven shapes in one
        # captured launch set, last two axes in plane tiles; new data is
        # copied into the bound buffer before each pass.
        dict(name="batch-256", kind="batch", mix="five", count=256, ndim=3, shapes=4, precision="c64", direction=-1,
             tile="planes", via="graph"),
        # A few complex-double inverse transforms with longer axes and mixed
        # radices, default schedule, plain launches.
        dict(name="batch-c128-back", kind="batch", count=24, lo=32, hi=256, step=16, ndim=3, shapes=9,
             precision="c128", direction=1, tile="full", via="run"),
        # The request loop: mixed shapes, precisions and directions from
        # pinned host buffers and back.
        dict(name="serve-24", kind="serve", count=24, lo=32, hi=256, step=16, shapes=5),
    ]


# ---------------------------------------------------------------- drawing

def _smooth(n):
    for p in (2, 3, 5, 7, 11, 13):
        while n % p == 0:
            n //= p
    return n == 1


def _length(rng, lo, hi, primes=False):
    """An axis length, spread over the logarithm: products of small primes
    (multiples of eight, odd ones and others), now and then any number."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.random()
    if primes and kind < 0.15:
        return n
    while n > lo:
        if _smooth(n) and (kind >= 0.75 or (n % 2 == 1 if kind >= 0.5 else n % 8 == 0)):
            return n
        n -= 1
    return lo


def _lengths(rng, ndim, lo, hi, points, primes=False):
    while True:
        v = [_length(rng, lo, hi, primes) for _ in range(ndim)]
        total = math.prod(v)
        if total <= points and (all(_smooth(n) for n in v) or (total <= 1 << 21 and max(v) <= 128)):
            return v


def _blocks_full(n, p):
    return -(-n // p) * (p - 1) < n


def _rank_grid(rng, shape, ranks):
    """A random factorisation of `ranks` over the axes that leaves no rank
    without coordinates; None when there is none."""
    for _ in range(40):
        g = [1] * len(shape)
        r = ranks
        for p in (2, 2, 2, 2, 2, 3):
            if r % p == 0:
                r //= p
                g[rng.randrange(len(shape))] *= p
        if all(_blocks_full(n, k) for n, k in zip(shape, g)):
            return g
    return None


def _join(v):
    return "x".join(str(int(a)) for a in v)


def _ints(text):
    return [int(a) for a in text.split("x")]


def draw(rng):
    kind = rng.choice(["split", "split", "split", "phases", "pencil", "reshape", "reshape", "chain", "batch", "batch",
                       "serve"])
    while True:
        c = _draw_kind(kind, rng)
        if c is not None:
            return c


def _draw_kind(kind, rng):
    prec = rng.choice(["c128", "c64"])
    if kind in ("split", "phases"):
        flat = rng.random() < 0.25
        points = 1 << rng.choice([13, 16, 19, 22, 25])
        shape = _lengths(rng, 2, 16, 4096, points, True) if flat else _lengths(rng, 3, 8, 512, points, True)
        ranks = rng.choice([1, 2, 4, 6, 8, 12, 32])
        g = _rank_grid(rng, shape, ranks)
        if g is None:
            return None
        fac = ""
        if rng.random() < 0.4:
            b = [rng.choice([q for q in range(1, n + 1) if n % q == 0]) for n in shape]
            if all(q == 1 for q in b):
                return None
            fac = _join(b)
        c = dict(kind="split", shape=_join(shape), grid=_join(g), ranks=ranks, factors=fac, precision=prec,
                 mode="forward" if kind == "phases" else rng.choice(["forward", "step"]),
                 order="phases" if kind == "phases" else "fused")
        s = _Split(c)
        if any(0 in lay.counts(r) for lay in (s.start, s.a, s.b) for r in range(lay.used)):
            return None
        return c
    if kind == "pencil":
        shape = _lengths(rng, 3, 16, 320, 1 << 24)
        g = rng.choice([(1, 2), (2, 2), (2, 3), (2, 4), (4, 8)])
        if any(not _blocks_full(n, p) for n in shape for p in g):
            return None
        return dict(kind="pencil", shape=_join(shape), grid=_join(g), ranks=g[0] * g[1], precision=prec)
    if kind == "reshape":
        shape = [max(8, int(math.exp(rng.uniform(math.log(10), math.log(400))))) for _ in range(3)]
        ranks = rng.choice([2, 4, 6, 8, 12])
        g, h = _rank_grid(rng, shape, ranks), _rank_grid(rng, shape, ranks)
        form = rng.choice(["rotated", "block", "permuted", "interleave"])
        if g is None or h is None:
            return None
        if form == "interleave":
            shape[0] = shape[0] // 4 * 4
            h = [4, h[1], 1]
            ranks = max(ranks, 4 * h[1])
            if not _blocks_full(shape[1], h[1]) or not _blocks_full(shape[0], g[0]):
                return None
        return dict(kind="reshape", shape=_join(shape), ranks=ranks, grid=_join(g), dest=_join(h), form=form,
                    words=rng.choice([1, 2, 3, 4, 6]))
    if kind == "chain":
        shape = [32 * rng.randint(2, 14) for _ in range(3)]
        return dict(kind="chain", shape=_join(shape), ranks=32, shift=_join([rng.randrange(n) for n in shape]))
    if kind == "batch":
        ndim = rng.choice([1, 2, 3, 3, 3])
        lo, hi = {1: (16, 4096), 2: (16, 512), 3: (16, 160)}[ndim]
        return dict(kind="batch", count=int(math.exp(rng.uniform(0, math.log(160)))), lo=lo, hi=hi,
                    step=rng.choice([1, 2, 8, 16]), ndim=ndim, shapes=rng.randrange(1000), precision=prec,
                    direction=rng.choice([-1, 1]), tile=rng.choice(["planes", "full"]), via=rng.choice(["graph", "run"]))
    return dict(kind="serve", count=rng.randint(2, 16), lo=16, hi=192, step=rng.choice([2, 8, 16]),
                shapes=rng.randrange(1000))


# ---------------------------------------------------------------- placement
# Where a decomposition puts a coordinate, from the descriptors' definitions.
# A descriptor is ("block", n, procs, factor), ("local", n), ("rotate",
# shift, nested), ("interleave", nested, B) or ("reverse", A, B, nested).

def _place(desc):
    """(processor position, local index) of every coordinate, processors."""
    kind = desc[0]
    if kind == "block":
        _, n, procs, factor = desc
        size = factor * max(1, -(-(n // factor) // procs))
        return [(g // size, g % size) for g in range(n)], procs
    if kind == "local":
        return [(0, g) for g in range(desc[1])], 1
    if kind == "rotate":
        inner, procs = _place(desc[2])
        n = len(inner)
        return [inner[(g + n + desc[1]) % n] for g in range(n)], procs
    if kind == "interleave":
        inner, procs = _place(desc[1])
        a = len(inner)
        return [(inner[g % a][0], g // a + desc[2] * inner[g % a][1]) for g in range(a * desc[2])], procs
    _, a, b, nested = desc
    inner, procs = _place(nested)
    return [inner[g // a + b * (g % a)] for g in range(a * b)], procs


def _make(C, desc):
    """The library's descriptor."""
    kind = desc[0]
    if kind == "block":
        return C.makeBlockDecomp(desc[1], desc[2])
    if kind == "local":
        return C.makeLocalDecomp(desc[1])
    nested = _make(C, desc[2] if kind == "rotate" else desc[1])
    made = C.makeRotatedDecomp(desc[1], nested) if kind == "rotate" else C.makeInterleaveDecomp(nested, desc[2])
    C.freeDimDecomp(nested)
    return made


class _Layout:
    """Descriptors on a rank grid.  strides: memory strides that every rank
    shares; without them each rank's block is packed in C order."""

    def __init__(self, descs, strides=None):
        self.descs, self.strides = descs, strides
        placed = [_place(d) for d in descs]
        self.procs = [p for _, p in placed]
        self.rank_stride = [math.prod(self.procs[i + 1:]) for i in range(len(descs))]
        self.used = math.prod(self.procs)
        self.own = []
        for table, procs in placed:
            mine = [[] for _ in range(procs)]
            for g, (p, off) in enumerate(table):
                mine[p].append((off, g))
            self.own.append([[g for _, g in sorted(m)] for m in mine])

    def coords(self, rank):
        return [self.own[i][rank // self.rank_stride[i] % self.procs[i]] for i in range(len(self.descs))]

    def counts(self, rank):
        return [len(c) for c in self.coords(rank)]

    def extent(self, rank):
        n = self.counts(rank)
        if 0 in n:
            return 0
        return 1 + sum((k - 1) * s for k, s in zip(n, self._strides(n)))

    def _strides(self, n):
        return self.strides or [math.prod(n[i + 1:]) for i in range(len(n))]

    def most(self):
        return max(self.extent(r) for r in range(self.used))

    def block(self, glob, rank, out=None):
        """Rank's local array of the global array (extra trailing axes are
        the element's words), zero where no coordinate sits."""
        nd = len(self.descs)
        words = glob.shape[nd:]
        if out is None:
            out = torch.zeros((self.extent(rank),) + tuple(words), dtype=glob.dtype, device=glob.device)
        part = glob
        for i, c in enumerate(self.coords(rank)):
            if c == list(range(c[0], c[0] + len(c))):
                part = part.narrow(i, c[0], len(c))
            else:
                part = part.index_select(i, torch.tensor(c, device=glob.device))
        n = self.counts(rank)
        w = math.prod(words) if words else 1
        strides = [s * w for s in self._strides(n)] + ([1] if words else [])
        out.view(-1).as_strided(tuple(n) + tuple(words), strides, out.storage_offset()).copy_(part)
        return out

    def make(self, C, comm):
        axes = [_make(C, d) for d in self.descs]
        if self.strides is None:
            return C.makePackedDecomp(comm, len(axes), dm.ptrs(axes))
        return C.makeDecomp(len(axes), dm.ptrs([C.makeAxisDecomp(comm, a, s, r) for a, s, r in
                                                zip(axes, self.strides, self.rank_stride)]))


def _grid_search(procs, tasks):
    """The processor grid of the reference's planner: least load, then the
    squarest, in its enumeration order (processor_grid.c:24-97)."""
    nd = len(tasks)
    best = dict(load=math.prod(tasks), asym=10000.0, grid=[1] * nd)

    def search(d, grid, used, load, mn, mx):
        now, k = used, 1
        while k <= procs and k <= tasks[d] and now <= procs:
            now = used * k
            if now <= procs:
                lo, hi = tasks[d] // k, -(-tasks[d] // k)
                total = load * hi
                lo, hi = min(mn, lo), max(mx, hi)
                if d < nd - 1:
                    search(d + 1, grid + [k], now, total, lo, hi)
                elif total < best["load"] or (total == best["load"] and hi / lo < best["asym"]):
                    best.update(load=total, asym=hi / lo, grid=grid + [k])
            k += 1
    search(0, [], 1, 1, max(tasks), 0)
    return best["grid"]


class _Split:
    """Start, first-stage and output layouts of a split-transform case."""

    def __init__(self, c):
        self.shape, self.grid = _ints(c["shape"]), _ints(c["grid"])
        self.n = math.prod(self.shape)
        if c["factors"]:
            self.B = _ints(c["factors"])
        else:  # the default split: A the largest divisor not above the root
            self.B = [n // max(q for q in range(1, n + 1) if n % q == 0 and q * q <= n) for n in self.shape]
        self.A = [n // b for n, b in zip(self.shape, self.B)]
        self.start = _Layout([("block", n, g, 1) for n, g in zip(self.shape, self.grid)])
        ga, gb = _grid_search(c["ranks"], self.A), _grid_search(c["ranks"], self.B)
        self.a = _Layout([("interleave", ("block", a, g, 1), b) for a, g, b in zip(self.A, ga, self.B)])
        blocked = [("block", a * b, g, a) for a, b, g in zip(self.A, self.B, gb)]
        self.b = _Layout([("reverse", b, a, d) for a, b, d in zip(self.A, self.B, blocked)])
        self.out = self.a if all(a == 1 for a in self.A) else self.b
        # a last stage alone writes the same layout; the first alone its own
        self.extent = max(self.a.most(), self.b.most() if any(a > 1 for a in self.A) else 0)


# ---------------------------------------------------------------- state

class _State:
    """What a program keeps between calls; releases the library's objects."""

    def __init__(self):
        self.undo, self.keep = [], []

    def later(self, f, *args):
        self.undo.append((f, args))

    def __del__(self):
        torch.cuda.synchronize()
        for f, args in reversed(self.undo):
            f(*args)


_lib = None
_stream = None


def _begin():
    """The library, and the one stream on which this program's torch work
    and its asynchronous library calls are ordered."""
    global _lib, _stream
    if _lib is None:
        _lib = dm.lib()
        _stream = torch.cuda.Stream()
    return _lib


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _field(shape, seed, dtype):
    """Uniform in [-1, 1), real and imaginary part."""
    real = torch.float64 if dtype == torch.complex128 else torch.float32
    x = torch.rand(tuple(shape) + (2,), generator=_gen(seed), device=DEV, dtype=real)
    return torch.view_as_complex(x.mul_(2).sub_(1))


def _buffer(C, s, comm, ranks, elems, dtype, words=1):
    """A distributed buffer in torch memory: one slot per rank."""
    t = torch.zeros((ranks, elems * words), dtype=dtype, device=DEV)
    if C.dm_register(comm, t.data_ptr(), elems * words * t.element_size()) != 0:
        raise RuntimeError("dm_register failed")
    s.later(C.dm_unregister, t.data_ptr())
    s.keep.append(t)
    return t


def _world(C, s, ranks, asynchronous):
    comm = C.dm_world_create(ranks)
    s.later(C.dm_world_free, comm)
    if asynchronous:
        C.dm_set_stream(comm, _stream.cuda_stream)
        C.dm_set_async(comm, 1)
    return comm


def _decomp(C, s, comm, layout):
    d = layout.make(C, comm)
    if not d:
        raise RuntimeError("no decomposition")
    s.later(C.freeDecomp, d)
    return d


def _scatter(layout, glob, buf, words=1):
    for r in range(layout.used):
        layout.block(glob, r, buf[r, :layout.extent(r) * words].view((-1, words) if words > 1 else (-1,)))


def prepare(case, seed):
    C = _begin()
    s = _State()
    s.case = case
    {"split": _prepare_split, "pencil": _prepare_pencil, "reshape": _prepare_reshape, "chain": _prepare_chain,
     "batch": _prepare_batch, "serve": _prepare_serve}[case["kind"]](C, s, case, seed)
    torch.cuda.synchronize()
    return s


def run(s):
    return s.pass_()


def _prepare_split(C, s, c, seed):
    sp = _Split(c)
    dtype = CDT[c["precision"]]
    comm = _world(C, s, c["ranks"], c["mode"] == "step")
    start = _decomp(C, s, comm, sp.start)
    dat = _buffer(C, s, comm, c["ranks"], sp.start.most(), dtype)
    length = 2 * sp.extent
    work = _buffer(C, s, comm, c["ranks"], length, dtype)
    f = "" if dtype == torch.complex128 else "f"
    if c["factors"]:
        plan = getattr(C, "makeParallelPlan" + f)(start, dm.ints(sp.B), dat.data_ptr(), length, work.data_ptr())
    else:
        plan = getattr(C, "makeSplitPlan" + f)(0, start, dat.data_ptr(), length, work.data_ptr())
    if not plan:
        raise RuntimeError("no plan")
    s.later(C.freeSplitPlan, plan)
    if c["order"] == "phases" and C.dm_split_set_phase_order(plan, 1) != 0:
        raise RuntimeError("no phase order")
    x = _field(sp.shape, seed, dtype)
    if c["mode"] == "backward":
        _scatter(sp.out, x, work)
    else:
        _scatter(sp.start, x, dat)
    result = [dat[r, :sp.start.extent(r)] for r in range(sp.start.used)]
    spectrum = [work[r, :sp.out.extent(r)] for r in range(sp.out.used)]
    if c["mode"] == "forward":
        def one():
            C.runSplitPlan(plan, dm.FFTW_FORWARD)
            return spectrum
    elif c["mode"] == "backward":
        def one():
            C.runSplitPlan(plan, dm.FFTW_BACKWARD)
            return result
    else:
        half = work[:, :sp.extent]

        def one():
            with torch.cuda.stream(_stream):
                C.runSplitPlan(plan, dm.FFTW_FORWARD)
                half.mul_(1.0 / sp.n)
                C.runSplitPlan(plan, dm.FFTW_BACKWARD)
            return result
    s.pass_ = one


def _pencil_layouts(c):
    shape, g = _ints(c["shape"]), _ints(c["grid"])

    def pencil(axis):
        left = iter(g)
        return _Layout([("local", n) if d == axis else ("block", n, next(left), 1) for d, n in enumerate(shape)])
    return shape, [pencil(0), pencil(1), pencil(2)]


def _prepare_pencil(C, s, c, seed):
    shape, (px, py, pz) = _pencil_layouts(c)
    dtype = CDT[c["precision"]]
    comm = _world(C, s, c["ranks"], True)
    dx, dy, dz = (_decomp(C, s, comm, p) for p in (px, py, pz))
    per = max(p.most() for p in (px, py, pz))
    b0, b1, b2 = (_buffer(C, s, comm, c["ranks"], per, dtype) for _ in range(3))
    double = 1 if dtype == torch.complex128 else 0
    stages = [(C.dm_plan_axis_fft(dx, dy, 0, double, dm.FFTW_FORWARD), b0.data_ptr(), b1.data_ptr()),
              (C.dm_plan_axis_fft(dy, dz, 1, double, dm.FFTW_FORWARD), b1.data_ptr(), b2.data_ptr()),
              (C.dm_plan_axis_fft(dz, dz, 2, double, dm.FFTW_FORWARD), b2.data_ptr(), b1.data_ptr())]
    for p, _, _ in stages:
        s.later(C.dm_free_axis_fft, p)
    _scatter(px, _field(shape, seed, dtype), b0)
    out = [b1[r, :pz.extent(r)] for r in range(pz.used)]

    def one():
        for p, src, dst in stages:
            C.dm_run_axis_fft(p, src, dst)
        return out
    s.pass_ = one


def _words(shape, words, seed):
    return torch.randint(-2 ** 31, 2 ** 31 - 1, tuple(shape) + ((words,) if words > 1 else ()), generator=_gen(seed),
                         device=DEV, dtype=torch.int32)


def _reshape_layouts(c):
    shape, g, h = _ints(c["shape"]), _ints(c["grid"]), _ints(c["dest"])
    src = _Layout([("block", n, p, 1) for n, p in zip(shape, g)])
    descs = [("block", n, p, 1) for n, p in zip(shape, h)]
    strides = None
    if c["form"] == "rotated":
        descs = [("rotate", n // 3, d) for n, d in zip(shape, descs)]
    if c["form"] in ("rotated", "permuted"):  # memory order: last axis slowest, then the first, the middle fastest
        most = [-(-n // p) for n, p in zip(shape, h)]
        strides = [most[1], 1, most[1] * most[0]]
    if c["form"] == "interleave":
        descs[0] = ("interleave", ("block", 4, 4, 1), shape[0] // 4)
    return shape, src, _Layout(descs, strides)


def _prepare_reshape(C, s, c, seed):
    shape, src, dst = _reshape_layouts(c)
    w = c["words"]
    comm = _world(C, s, c["ranks"], False)
    ds, dd = _decomp(C, s, comm, src), _decomp(C, s, comm, dst)
    base = ctypes.c_void_p()
    C.dm_type_contiguous(w, dm.mpi_type("int"), ctypes.byref(base))
    s.later(C.dm_type_free, ctypes.byref(base))
    plan = C.makeReshapePlan(comm, base, ds, dd)
    if not plan:
        raise RuntimeError("no plan")
    s.later(C.freeReshapePlan, plan)
    a = _buffer(C, s, comm, c["ranks"], src.most(), torch.int32, w)
    b = _buffer(C, s, comm, c["ranks"], dst.most(), torch.int32, w)
    _scatter(src, _words(shape, w, seed), a, w)
    out = [b[r, :dst.extent(r) * w] for r in range(dst.used)]
    pa, pb = a.data_ptr(), b.data_ptr()

    def one():
        C.runReshapePlan(comm, plan, pa, pb)
        return out
    s.pass_ = one


def _chain_layouts(c):
    shape, shift = _ints(c["shape"]), _ints(c["shift"])
    n0, n1, n2 = shape
    block = _Layout([("block", n0, 4, 1), ("block", n1, 8, 1), ("local", n2)], [n1 // 8 * n2, n2, 1])
    rot = _Layout([("rotate", k, d) for k, d in zip(shift, block.descs)], [n1 // 8, 1, n0 // 4 * (n1 // 8)])
    inter = _Layout([("interleave", ("block", 4, 4, 1), n0 // 4), ("block", n1, 8, 1), ("local", n2)])
    return shape, block, rot, inter


def _prepare_chain(C, s, c, seed):
    shape, block, rot, inter = _chain_layouts(c)
    comm = _world(C, s, c["ranks"], False)
    d = [_decomp(C, s, comm, x) for x in (block, rot, inter)]
    t = dm.mpi_type("long_long")
    plans = [C.makeReshapePlan(comm, t, d[0], d[1]), C.makeReshapePlan(comm, t, d[1], d[2])]
    if not all(plans):
        raise RuntimeError("no plan")
    for p in plans:
        s.later(C.freeReshapePlan, p)
    bufs = [_buffer(C, s, comm, c["ranks"], x.most(), torch.int64) for x in (block, rot, inter)]
    glob = torch.randint(-2 ** 62, 2 ** 62, tuple(shape), generator=_gen(seed), device=DEV, dtype=torch.int64)
    _scatter(block, glob, bufs[0])
    at = [b.data_ptr() for b in bufs]

    def one():
        C.runReshapePlan(comm, plans[0], at[0], at[1])
        C.runReshapePlan(comm, plans[1], at[1], at[2])
        return bufs[1:]
    s.pass_ = one


def _shapes(c):
    """Transform shapes of a batch or request list: the seeded batch of the
    package's workloads (mix "five": each axis from {32, 48, 64, 96, 128}),
    or axes log-uniform in [lo, hi], rounded to a multiple of step (any
    length when step is 1: products of primes up to 13)."""
    if c.get("mix") == "five":
        return [list(v) for v in workloads.batched_shapes(c["count"], c["shapes"])]
    rng = random.Random(1000 + c["shapes"])
    out, total = [], 0
    for _ in range(c["count"]):
        v = []
        for _ in range(c.get("ndim", 3)):
            n = math.exp(rng.uniform(math.log(c["lo"]), math.log(c["hi"])))
            n = int(round(n / c["step"])) * c["step"]
            while not _smooth(n):
                n -= c["step"] if c["step"] > 1 and n > c["lo"] + c["step"] else 1
            v.append(min(c["hi"], max(c["lo"], n)))
        if out and total + math.prod(v) > 1 << 27:  # a batch of at most 1 GiB of complex floats
            break
        out.append(v)
        total += math.prod(v)
    return out


def _batch_parts(c):
    shapes = _shapes(c)
    offs, at = [], 0
    for v in shapes:  # 256-byte aligned, as an allocator gives them
        offs.append(at)
        at += -(-math.prod(v) // 32) * 32
    return shapes, offs, at


def _prepare_batch(C, s, c, seed):
    shapes, offs, total = _batch_parts(c)
    dtype = CDT[c["precision"]]
    es = torch.empty(0, dtype=dtype).element_size()
    x = _field([total], seed, dtype)
    buf = torch.empty_like(x)
    plan = C.dm_batch_plan(len(shapes), c["ndim"], dm.ints([n for v in shapes for n in v]),
                           1 if dtype == torch.complex128 else 0, c["direction"])
    if not plan:
        raise RuntimeError("no plan")
    s.later(C.dm_batch_free, plan)
    s.keep += [x, buf]
    if c["tile"] == "planes":
        C.dm_batch_set_schedule(plan, dm.DM_BATCH_TILE_PLANES, 0)
    if C.dm_batch_bind(plan, dm.ptrs([buf.data_ptr() + o * es for o in offs])) != 0:
        raise RuntimeError("dm_batch_bind failed")
    call = C.dm_batch_graph_launch if c["via"] == "graph" else C.dm_batch_run
    at = _stream.cuda_stream
    # one tensor per transform while they are few, else the whole buffer
    out = [buf[o:o + math.prod(v)] for v, o in zip(shapes, offs)] if len(shapes) <= 60 else buf

    def one():
        with torch.cuda.stream(_stream):
            buf.copy_(x)
            if call(plan, at) != 0:
                raise RuntimeError("batch failed")
        return out
    s.pass_ = one


def _requests(c):
    rng = random.Random(c["shapes"])
    return [(v, "c64" if rng.random() < 0.7 else "c128", rng.choice([-1, 1])) for v in _shapes(dict(c, ndim=3))]


def _prepare_serve(C, s, c, seed):
    reqs = []
    server = C.dm_server_create(64 << 30, 4, 8)
    if not server:
        raise RuntimeError("no server")
    s.later(C.dm_server_destroy, server)
    outs = []
    for k, (v, prec, direction) in enumerate(_requests(c)):
        x = torch.empty(v, dtype=CDT[prec], pin_memory=True)
        y = torch.empty(v, dtype=CDT[prec], pin_memory=True)
        x.copy_(_field(v, seed * 1000 + k, CDT[prec]))
        s.keep += [x, y]
        outs.append(y)
        reqs.append((3, dm.ints(v), 1 if prec == "c128" else 0, direction, x.data_ptr(), y.data_ptr()))

    def one():
        for r in reqs:
            if C.dm_server_submit(server, *r) < 0:
                raise RuntimeError("request refused")
            C.dm_server_poll(server)
        C.dm_server_drain(server)
        return outs
    s.pass_ = one


# ---------------------------------------------------------------- work, exact

def work(case):
    c = case
    if c["kind"] in ("split", "pencil"):
        n = math.prod(_ints(c["shape"]))
        es = 16 if c["precision"] == "c128" else 8
        times = 2 if c.get("mode") == "step" else 1
        return {"bytes": 2 * n * es, "flops": times * 5 * n * math.log2(n)}
    if c["kind"] == "reshape":
        return {"bytes": 2 * math.prod(_ints(c["shape"])) * 4 * c["words"], "flops": 0}
    if c["kind"] == "chain":  # two hops, both results returned
        return {"bytes": 3 * math.prod(_ints(c["shape"])) * 8, "flops": 0}
    if c["kind"] == "batch":
        sizes = [(math.prod(v), c["precision"]) for v in _shapes(c)]
    else:
        sizes = [(math.prod(v), prec) for v, prec, _ in _requests(c)]
    return {"bytes": sum(2 * n * (16 if p == "c128" else 8) for n, p in sizes),
            "flops": sum(5 * n * math.log2(max(2, n)) for n, _ in sizes)}


def _dft(x, direction=-1):
    """The unnormalised transform over all axes, in 64 bits."""
    x = x.to(torch.complex128)
    if x.numel() <= 1 << 23:
        x = x.cpu()
    y = torch.fft.fftn(x) if direction == -1 else torch.fft.ifftn(x, norm="forward")
    return y.to(DEV)


def exact(case, seed):
    c = case
    if c["kind"] == "split":
        sp = _Split(c)
        x = _field(sp.shape, seed, CDT[c["precision"]])
        if c["mode"] == "forward":
            x = _dft(x)
            return [sp.out.block(x, r) for r in range(sp.out.used)]
        if c["mode"] == "backward":
            x = _dft(x, 1)
        return [sp.start.block(x, r) for r in range(sp.start.used)]
    if c["kind"] == "pencil":
        shape, (_, _, pz) = _pencil_layouts(c)
        x = _dft(_field(shape, seed, CDT[c["precision"]]))
        return [pz.block(x, r) for r in range(pz.used)]
    if c["kind"] == "reshape":
        shape, _, dst = _reshape_layouts(c)
        x = _words(shape, c["words"], seed)
        return [dst.block(x, r).view(-1) for r in range(dst.used)]
    if c["kind"] == "chain":
        shape, _, rot, inter = _chain_layouts(c)
        glob = torch.randint(-2 ** 62, 2 ** 62, tuple(shape), generator=_gen(seed), device=DEV, dtype=torch.int64)
        return [torch.stack([lay.block(glob, r) for r in range(lay.used)]) for lay in (rot, inter)]
    if c["kind"] == "batch":
        shapes, offs, total = _batch_parts(c)
        x = _field([total], seed, CDT[c["precision"]])
        y = x.to(torch.complex128)
        for v, o in zip(shapes, offs):
            n = math.prod(v)
            y[o:o + n] = _dft(x[o:o + n].view(v), c["direction"]).reshape(-1)
        return [y[o:o + math.prod(v)] for v, o in zip(shapes, offs)] if len(shapes) <= 60 else y
    return [_dft(_field(v, seed * 1000 + k, CDT[prec]), direction).cpu()
            for k, (v, prec, direction) in enumerate(_requests(c))]
