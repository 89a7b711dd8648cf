// K1: decomposition-driven reshape as a device gather.
//
// The reference moves each rank's share as MPI messages built from nested
// indexed datatypes (reshape.c:461-492, typelist.c:74-106).  Here every
// virtual rank's local array is a slot of one HBM buffer, so a reshape is
// one launch: each global coordinate is read from its source owner's slot
// and written to its destination owner's slot.  Placement is given by
// per-axis lookup tables (owner contribution and local offset per global
// coordinate) plus per-rank memory strides.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "kernels.h"

namespace dm {

namespace {

constexpr int TILE = 32;      // tile edge (elements)
constexpr int ROWS = 8;       // thread rows per tile pass
constexpr int NTHREADS = TILE * ROWS;
// Batch slices per 2D-tile workgroup: 2 (16 KiB of 8-byte elements; 4
// measured 5% slower, 1 20%), 1 for 16-byte elements (the same 16 KiB:
// 2.09 / 2.05 -> 2.00 / 1.96 ms per step for the phase-order reshapes).
constexpr int tile_slices(int bytes) { return bytes >= 16 ? 1 : 2; }

template <int BYTES>
struct Elem;
template <> struct Elem<1> { typedef uint8_t T; };
template <> struct Elem<2> { typedef uint16_t T; };
template <> struct Elem<4> { typedef uint32_t T; };
template <> struct Elem<8> { typedef uint64_t T; };
template <> struct Elem<16> { typedef unsigned int T __attribute__((ext_vector_type(4))); };

// 12- and 24-byte elements (three floats, three doubles) move whole: as three
// separate words each access would use a third of its lines.
struct E12 { uint32_t x, y, z; };
struct E24 { uint64_t x, y, z; };
template <> struct Elem<12> { typedef E12 T; };
template <> struct Elem<24> { typedef E24 T; };

// One element access.  NT: the non-temporal hint (a template argument: a
// hinted and a plain access in two branches are merged into one by the
// compiler, which drops the hint).
template <bool NT, typename E>
__device__ __forceinline__ E take(const E *e) {
  if constexpr (!NT) return *e;
  else if constexpr (sizeof(E) == 12 || sizeof(E) == 24)
    return {__builtin_nontemporal_load(&e->x), __builtin_nontemporal_load(&e->y), __builtin_nontemporal_load(&e->z)};
  else return __builtin_nontemporal_load(e);
}
template <bool NT, typename E>
__device__ __forceinline__ void give(E *e, E v) {
  if constexpr (!NT) {
    *e = v;
  } else if constexpr (sizeof(E) == 12 || sizeof(E) == 24) {
    __builtin_nontemporal_store(v.x, &e->x);
    __builtin_nontemporal_store(v.y, &e->y);
    __builtin_nontemporal_store(v.z, &e->z);
  } else {
    __builtin_nontemporal_store(v, e);
  }
}

// Per-block partial sums of the batch axes for one layout.
struct Partial {
  int rank;
  i64 addr;                   // uniform strides: sum of m_d * off_d
  int off[DM_MAX_DIMS];       // non-uniform: the batch axes' local offsets
};

// Batch part of a workgroup's coordinates: batch index bidx decoded over
// the batch axes (last batch axis fastest) straight into the sums, so no
// coordinate array is indexed at run time.
template <bool UNIFORM>
__device__ __forceinline__ void partial_init(const DevLayout &Lt, const ReshapeLaunch &p, long long bidx,
                                             Partial &q) {
  q.rank = 0;
  q.addr = 0;
  for (int k = p.nbatch - 1; k >= 0; k--) {
    int d = p.batch_axis[k];
    int g = (int)(bidx % p.L[d]);
    bidx /= p.L[d];
    q.rank += Lt.rank[Lt.at[d] + g];
    if (UNIFORM) q.addr += Lt.addr[Lt.at[d] + g];
    else q.off[k] = Lt.off[Lt.at[d] + g];
  }
}

// Element offset (in elements, from slot 0) of the coordinate whose batch
// part is q and whose tile axes take values ga (axis a) and gb (axis b);
// returns -1 when the owner rank is outside the layout's ranks.
template <bool UNIFORM>
__device__ __forceinline__ i64 locate(const DevLayout &Lt, const ReshapeLaunch &p, const Partial &q,
                                      int a, int ga, int b, int gb, i64 slot) {
  int R = q.rank + Lt.rank[Lt.at[a] + ga] + (b != a ? Lt.rank[Lt.at[b] + gb] : 0);
  if (R >= Lt.proc_used) return -1;
  i64 off;
  if (UNIFORM) {
    off = q.addr + Lt.addr[Lt.at[a] + ga] + (b != a ? Lt.addr[Lt.at[b] + gb] : 0);
  } else {
    const i64 *m = Lt.strides + (i64)R * Lt.ndim;
    off = m[a] * Lt.off[Lt.at[a] + ga];
    if (b != a) off += m[b] * Lt.off[Lt.at[b] + gb];
    for (int k = 0; k < p.nbatch; k++) off += m[p.batch_axis[k]] * q.off[k];
  }
  return (i64)R * slot + off;
}

// 2D tile: read rows along b (source-contiguous), write rows along a.
// A workgroup moves NB tiles that differ only in the batch coordinate (so
// the tile-axis tables are shared and more bytes are in flight per
// workgroup).  Each side runs in three branch-free phases: every address of
// the thread's elements (table loads only), then every data load (clamped
// to element 0 of the region when the element is absent), then the LDS (or
// global) writes.  A load queue that completes in order would otherwise
// stall each data load behind the next element's table loads.
template <int BYTES, bool US, bool UD, int NB, bool NT>
__global__ __launch_bounds__(NTHREADS) void reshape_tile2d(ReshapeLaunch p) {
  typedef typename Elem<BYTES>::T E;
  constexpr int RPT = TILE / ROWS;
  __shared__ E tile[NB][TILE][TILE + 1];
  __shared__ unsigned char have[NB][TILE][TILE + 1];

  long long bid = blockIdx.x;
  int ta = (int)(bid % p.tiles_a);
  bid /= p.tiles_a;
  int tb = (int)(bid % p.tiles_b);
  bid /= p.tiles_b;
  Partial qs[NB], qd[NB];
  bool live[NB];
#pragma unroll
  for (int n = 0; n < NB; n++) {
    long long b = bid * NB + n;
    live[n] = b < p.nbatch_total;
    partial_init<US>(p.src, p, live[n] ? b : 0, qs[n]);
    partial_init<UD>(p.dst, p, live[n] ? b : 0, qd[n]);
  }

  const E *src = reinterpret_cast<const E *>(p.src_base);
  E *dst = reinterpret_cast<E *>(p.dst_base);
  const int La = p.L[p.a], Lb = p.L[p.b];
  int a0 = ta * TILE, b0 = tb * TILE;
  int tx = threadIdx.x % TILE, ty = threadIdx.x / TILE;

  // load: consecutive threads walk axis b
  i64 s[NB][RPT];
  if constexpr (US) {
    // uniform source: the tile axes' table entries are loaded once (one per
    // column, one per row) and shared by the NB slices
    const int gbc = min(b0 + tx, Lb - 1);
    const int rb = p.src.rank[p.src.at[p.b] + gbc];
    const i64 ab = p.src.addr[p.src.at[p.b] + gbc];
    int ra[RPT];
    i64 aa[RPT];
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int gac = min(a0 + ty + k * ROWS, La - 1);
      ra[k] = p.src.rank[p.src.at[p.a] + gac];
      aa[k] = p.src.addr[p.src.at[p.a] + gac];
    }
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
      for (int k = 0; k < RPT; k++) {
        const bool in = live[n] && a0 + ty + k * ROWS < La && b0 + tx < Lb;
        const int R = qs[n].rank + ra[k] + rb;
        s[n][k] = (in && R < p.src.proc_used) ? (i64)R * p.src_slot + qs[n].addr + aa[k] + ab : -1;
      }
  } else {
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
      for (int k = 0; k < RPT; k++) {
        int ga = a0 + ty + k * ROWS, gb = b0 + tx;
        bool in = live[n] && ga < La && gb < Lb;
        s[n][k] = locate<US>(p.src, p, qs[n], p.a, in ? ga : 0, p.b, in ? gb : 0, p.src_slot);
        if (!in) s[n][k] = -1;
      }
  }
  E v[NB][RPT];
#pragma unroll
  for (int n = 0; n < NB; n++)
#pragma unroll
    for (int k = 0; k < RPT; k++) v[n][k] = take<NT>(src + (s[n][k] >= 0 ? s[n][k] : 0));
#pragma unroll
  for (int n = 0; n < NB; n++)
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      tile[n][ty + k * ROWS][tx] = v[n][k];
      have[n][ty + k * ROWS][tx] = s[n][k] >= 0;
    }
  __syncthreads();
  // store: consecutive threads walk axis a
  i64 d[NB][RPT];
  if constexpr (UD) {
    const int gac = min(a0 + tx, La - 1);
    const int ra = p.dst.rank[p.dst.at[p.a] + gac];
    const i64 aa = p.dst.addr[p.dst.at[p.a] + gac];
    int rb[RPT];
    i64 ab[RPT];
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int gbc = min(b0 + ty + k * ROWS, Lb - 1);
      rb[k] = p.dst.rank[p.dst.at[p.b] + gbc];
      ab[k] = p.dst.addr[p.dst.at[p.b] + gbc];
    }
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
      for (int k = 0; k < RPT; k++) {
        const bool in = live[n] && a0 + tx < La && b0 + ty + k * ROWS < Lb && have[n][tx][ty + k * ROWS];
        const int R = qd[n].rank + ra + rb[k];
        d[n][k] = (in && R < p.dst.proc_used) ? (i64)R * p.dst_slot + qd[n].addr + aa + ab[k] : -1;
      }
  } else {
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
      for (int k = 0; k < RPT; k++) {
        int ga = a0 + tx, gb = b0 + ty + k * ROWS;
        bool in = live[n] && ga < La && gb < Lb;
        d[n][k] = locate<UD>(p.dst, p, qd[n], p.a, in ? ga : 0, p.b, in ? gb : 0, p.dst_slot);
        if (!in || !have[n][tx][ty + k * ROWS]) d[n][k] = -1;
      }
  }
#pragma unroll
  for (int n = 0; n < NB; n++)
#pragma unroll
    for (int k = 0; k < RPT; k++)
      if (d[n][k] >= 0) give<NT>(dst + d[n][k], tile[n][tx][ty + k * ROWS]);
}

// 1D runs along axis a (same fastest axis on both sides), phased as above.
template <int BYTES, bool US, bool UD, bool NT>
__global__ __launch_bounds__(NTHREADS) void reshape_run1d(ReshapeLaunch p) {
  typedef typename Elem<BYTES>::T E;
  constexpr int PER = 4;
  long long bid = blockIdx.x;
  int ta = (int)(bid % p.tiles_a);
  bid /= p.tiles_a;
  Partial qs, qd;
  partial_init<US>(p.src, p, bid, qs);
  partial_init<UD>(p.dst, p, bid, qd);
  const E *src = reinterpret_cast<const E *>(p.src_base);
  E *dst = reinterpret_cast<E *>(p.dst_base);
  const int La = p.L[p.a];
  int base = ta * NTHREADS * PER;
  i64 s[PER], d[PER];
#pragma unroll
  for (int k = 0; k < PER; k++) {
    int ga = base + k * NTHREADS + threadIdx.x;
    bool in = ga < La;
    int g = in ? ga : 0;
    s[k] = locate<US>(p.src, p, qs, p.a, g, p.a, g, p.src_slot);
    d[k] = locate<UD>(p.dst, p, qd, p.a, g, p.a, g, p.dst_slot);
    if (!in || s[k] < 0 || d[k] < 0) s[k] = d[k] = -1;
  }
  E v[PER];
#pragma unroll
  for (int k = 0; k < PER; k++) v[k] = take<NT>(src + (s[k] >= 0 ? s[k] : 0));
#pragma unroll
  for (int k = 0; k < PER; k++)
    if (d[k] >= 0) give<NT>(dst + d[k], v[k]);
}

// ---- every coordinate owned on both sides ----------------------------------

// f(axis, coordinate) for every batch axis at batch index bidx (last batch
// axis fastest); 32-bit divisions while the index fits.
template <typename F>
__device__ __forceinline__ void batch_walk(const ReshapeLaunch &p, long long bidx, F f) {
  if (p.nbatch_total < (1LL << 31)) {
    unsigned b = (unsigned)bidx;
    for (int k = p.nbatch - 1; k >= 0; k--) {
      const int d = p.batch_axis[k];
      const unsigned l = (unsigned)p.L[d], q = b / l;
      f(d, (int)(b - q * l));
      b = q;
    }
  } else {
    for (int k = p.nbatch - 1; k >= 0; k--) {
      const int d = p.batch_axis[k];
      f(d, (int)(bidx % p.L[d]));
      bidx /= p.L[d];
    }
  }
}

// Byte offsets of one side's elements in a workgroup's tile.  OT: their
// type -- unsigned while both buffers are below 4 GiB: then a uniform base
// in scalar registers and one 32-bit add per element (512^3 int64 chain: 844 us
// against 882 with 64-bit sums).
// Uniform strides: the batch part goes into the base, an element adds its a
// part and its b part.  Otherwise the owners of the tile are pairs of
// positions (along a, along b), and LDS holds for each pair the batch part
// of the address and the strides along a and b, so that an element costs
// LDS reads and no table of its own.  (Forming it from the owner's strides
// in memory cost ndim + 2 loads an element: 79 us for 150 x 77 x 201
// 12-byte elements on 12 ranks.)
template <int BYTES, bool UNIFORM, int NB, typename OT>
struct SideAddr;

template <int BYTES, int NB, typename OT>
struct SideAddr<BYTES, true, NB, OT> {
  i64 batch[NB];
  typedef OT Part;
  __device__ __forceinline__ void init(const ReshapeSide &, const DevLayout &, const ReshapeLaunch &, long long, int n,
                                       char *, i64 slot, int rank, i64 addr) {
    batch[n] = (i64)rank * slot + addr * BYTES;
  }
  __device__ __forceinline__ Part part(const ReshapeSide &s, const DevLayout &L, int axis, int d, int g, i64 slot) const {
    if constexpr (sizeof(OT) == 4) {
      const uint2 q = *reinterpret_cast<const uint2 *>(s.part[axis] + 2 * (size_t)g);
      return q.x * (unsigned)slot + q.y * (unsigned)BYTES;
    } else {
      return (i64)L.rank[L.at[d] + g] * slot + L.addr[L.at[d] + g] * BYTES;
    }
  }
  __device__ __forceinline__ i64 base(int n) const { return batch[n]; }
  __device__ __forceinline__ OT at(const ReshapeSide &, int, Part a, Part b) const { return a + b; }
};

template <int BYTES, int NB, typename OT>
struct SideAddr<BYTES, false, NB, OT> {
  typedef __attribute__((address_space(3))) OT lds_ot;
  lds_ot *tab;  // per pair and slice: batch part, stride along a, stride along b
  struct Part {
    int pos;
    int off;
  };
  // rank: the batch coordinates' owner contribution
  __device__ __forceinline__ void init(const ReshapeSide &s, const DevLayout &L, const ReshapeLaunch &p,
                                       long long bidx, int n, char *lds, i64 slot, int rank, i64) {
    tab = (lds_ot *)(lds);
    const int pairs = s.np[0] * s.np[1];
    for (int e = threadIdx.x; e < pairs; e += (int)blockDim.x) {
      const int qa = e / s.np[1], qb = e - qa * s.np[1];
      const int R = rank + s.posrank[0][qa] + s.posrank[1][qb];
      const i64 *m = L.strides + (i64)R * L.ndim;
      i64 addr = 0;
      batch_walk(p, bidx, [&](int d, int g) { addr += m[d] * L.off[L.at[d] + g]; });
      lds_ot *q = tab + 3 * (e * NB + n);
      q[0] = (OT)((i64)R * slot + addr * BYTES);
      q[1] = (OT)(m[p.a] * BYTES);
      q[2] = (OT)(m[p.b] * BYTES);
    }
  }
  // axis: 0 for a, 1 for b
  __device__ __forceinline__ Part part(const ReshapeSide &s, const DevLayout &L, int axis, int d, int g, i64) const {
    return {s.pos[axis][g], L.off[L.at[d] + g]};
  }
  __device__ __forceinline__ i64 base(int) const { return 0; }
  __device__ __forceinline__ OT at(const ReshapeSide &s, int n, Part a, Part b) const {
    const lds_ot *q = tab + 3 * ((a.pos * s.np[1] + b.pos) * NB + n);
    return q[0] + (OT)a.off * q[1] + (OT)b.off * q[2];
  }
};

// Both sides' batch parts for slice n at batch index bidx.
template <int BYTES, bool US, bool UD, int NB, typename OT>
__device__ __forceinline__ void batch_parts(const ReshapeLaunch &p, long long bidx, int n,
                                            SideAddr<BYTES, US, NB, OT> &src, SideAddr<BYTES, UD, NB, OT> &dst,
                                            char *lds) {
  int rs = 0, rd = 0;
  i64 as = 0, ad = 0;
  batch_walk(p, bidx, [&](int d, int g) {
    rs += p.src.rank[p.src.at[d] + g];
    rd += p.dst.rank[p.dst.at[d] + g];
    if constexpr (US) as += p.src.addr[p.src.at[d] + g];
    if constexpr (UD) ad += p.dst.addr[p.dst.at[d] + g];
  });
  src.init(p.ss, p.src, p, bidx, n, lds, p.src_bytes, rs, as);
  dst.init(p.sd, p.dst, p, bidx, n, lds + (US ? 0 : p.ss.np[0] * p.ss.np[1] * 3 * NB * sizeof(OT)), p.dst_bytes, rd,
           ad);
}
template <bool US, bool UD, int NB, typename OT>
size_t side_lds(const ReshapeLaunch &p) {
  return ((US ? 0 : p.ss.np[0] * p.ss.np[1]) + (UD ? 0 : p.sd.np[0] * p.sd.np[1])) * 3 * NB * sizeof(OT);
}

// Tile transpose: TA values of axis a (the destination's fastest) x TB of
// axis b (the source's) x NB batch slices through LDS; lanes read along b
// and write along a.  Loads go out together, after every address.
template <int BYTES, bool US, bool UD, int TA, int TB, int NB, typename OT, bool NT>
__global__ __launch_bounds__(NTHREADS) void reshape_tile(ReshapeLaunch p) {
  typedef typename Elem<BYTES>::T E;
  constexpr int N = TA * TB / NTHREADS;        // elements per thread and slice
  constexpr int SB = NTHREADS / TB, SA = NTHREADS / TA;
  __shared__ E tile[NB][TA][TB + 1];
  extern __shared__ __align__(16) char lds[];                // the sides' pair tables
  long long bid = blockIdx.x;
  const int ta = (int)(bid % p.tiles_a);
  bid /= p.tiles_a;
  const int tb = (int)(bid % p.tiles_b);
  bid /= p.tiles_b;
  SideAddr<BYTES, US, NB, OT> src;
  SideAddr<BYTES, UD, NB, OT> dst;
  bool live[NB];
#pragma unroll
  for (int n = 0; n < NB; n++) {
    const long long b = bid * NB + n;
    live[n] = b < p.nbatch_total;
    batch_parts<BYTES, US, UD, NB, OT>(p, live[n] ? b : 0, n, src, dst, lds);
  }
  if constexpr (!US || !UD) __syncthreads();
  const int a0 = ta * TA, b0 = tb * TB, La = p.L[p.a], Lb = p.L[p.b];
  {
    const int tx = threadIdx.x % TB, ty = threadIdx.x / TB;
    const auto cb = src.part(p.ss, p.src, 1, p.b, min(b0 + tx, Lb - 1), p.src_bytes);
    OT at[NB][N];
#pragma unroll
    for (int k = 0; k < N; k++) {
      const auto ca = src.part(p.ss, p.src, 0, p.a, min(a0 + ty + k * SB, La - 1), p.src_bytes);
#pragma unroll
      for (int n = 0; n < NB; n++) at[n][k] = src.at(p.ss, n, ca, cb);
    }
    E v[NB][N];
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
      for (int k = 0; k < N; k++) v[n][k] = take<NT>(reinterpret_cast<const E *>(p.src_base + src.base(n) + at[n][k]));
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
      for (int k = 0; k < N; k++) tile[n][ty + k * SB][tx] = v[n][k];
  }
  const int tx = threadIdx.x % TA, ty = threadIdx.x / TA;
  const auto ca = dst.part(p.sd, p.dst, 0, p.a, min(a0 + tx, La - 1), p.dst_bytes);
  OT at[NB][N];
#pragma unroll
  for (int k = 0; k < N; k++) {
    const auto cb = dst.part(p.sd, p.dst, 1, p.b, min(b0 + ty + k * SA, Lb - 1), p.dst_bytes);
#pragma unroll
    for (int n = 0; n < NB; n++) at[n][k] = dst.at(p.sd, n, ca, cb);
  }
  __syncthreads();
  E v[NB][N];
#pragma unroll
  for (int n = 0; n < NB; n++)
#pragma unroll
    for (int k = 0; k < N; k++) v[n][k] = tile[n][tx][ty + k * SA];
#pragma unroll
  for (int n = 0; n < NB; n++)
#pragma unroll
    for (int k = 0; k < N; k++)
      if (live[n] && a0 + tx < La && b0 + ty + k * SA < Lb) 
        give<NT>(reinterpret_cast<E *>(p.dst_base + dst.base(n) + at[n][k]), v[n][k]);
}

// Both sides fastest along a: rows of TX lanes along a, N rows of axis b per
// thread, straight from load to store.  (One workgroup per row of up to 1024
// elements left most lanes of short rows idle.)
template <int BYTES, bool US, bool UD, int TX, typename OT, bool NT>
__global__ __launch_bounds__(NTHREADS) void reshape_rows(ReshapeLaunch p) {
  typedef typename Elem<BYTES>::T E;
  constexpr int N = BYTES >= 16 ? 4 : 8, SB = NTHREADS / TX;
  extern __shared__ __align__(16) char lds[];
  long long bid = blockIdx.x;
  const int ta = (int)(bid % p.tiles_a);
  bid /= p.tiles_a;
  const int tb = (int)(bid % p.tiles_b);
  bid /= p.tiles_b;
  SideAddr<BYTES, US, 1, OT> src;
  SideAddr<BYTES, UD, 1, OT> dst;
  batch_parts<BYTES, US, UD, 1, OT>(p, bid, 0, src, dst, lds);
  if constexpr (!US || !UD) __syncthreads();
  const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
  const int ga = ta * TX + tx, La = p.L[p.a], Lb = p.L[p.b], gac = min(ga, La - 1);
  const auto sa = src.part(p.ss, p.src, 0, p.a, gac, p.src_bytes);
  const auto da = dst.part(p.sd, p.dst, 0, p.a, gac, p.dst_bytes);
  OT from[N], to[N];
#pragma unroll
  for (int k = 0; k < N; k++) {
    const int gbc = min((tb * N + k) * SB + ty, Lb - 1);
    from[k] = src.at(p.ss, 0, sa, src.part(p.ss, p.src, 1, p.b, gbc, p.src_bytes));
    to[k] = dst.at(p.sd, 0, da, dst.part(p.sd, p.dst, 1, p.b, gbc, p.dst_bytes));
  }
  E v[N];
#pragma unroll
  for (int k = 0; k < N; k++) v[k] = take<NT>(reinterpret_cast<const E *>(p.src_base + src.base(0) + from[k]));
#pragma unroll
  for (int k = 0; k < N; k++)
    if (ga < La && (tb * N + k) * SB + ty < Lb) give<NT>(reinterpret_cast<E *>(p.dst_base + dst.base(0) + to[k]), v[k]);
}

template <int BYTES, bool US, bool UD, int TA, int TB, int NB>
hipError_t launch_tile(ReshapeLaunch &p, hipStream_t s) {
  p.tiles_a = (p.L[p.a] + TA - 1) / TA;
  p.tiles_b = (p.L[p.b] + TB - 1) / TB;
  p.nblocks = (long long)p.tiles_a * p.tiles_b * ((p.nbatch_total + NB - 1) / NB);
  if (p.nblocks <= 0) return hipSuccess;
  const dim3 grid((unsigned)p.nblocks), block(NTHREADS);
  const size_t l4 = side_lds<US, UD, NB, unsigned>(p), l8 = side_lds<US, UD, NB, i64>(p);
  if (p.below_4g && p.nontemporal)
    hipLaunchKernelGGL((reshape_tile<BYTES, US, UD, TA, TB, NB, unsigned, true>), grid, block, l4, s, p);
  else if (p.below_4g) hipLaunchKernelGGL((reshape_tile<BYTES, US, UD, TA, TB, NB, unsigned, false>), grid, block, l4, s, p);
  else if (p.nontemporal) hipLaunchKernelGGL((reshape_tile<BYTES, US, UD, TA, TB, NB, i64, true>), grid, block, l8, s, p);
  else hipLaunchKernelGGL((reshape_tile<BYTES, US, UD, TA, TB, NB, i64, false>), grid, block, l8, s, p);
  return hipGetLastError();
}
template <int BYTES, bool US, bool UD, int TX>
hipError_t launch_rows(ReshapeLaunch &p, hipStream_t s) {
  constexpr int N = BYTES >= 16 ? 4 : 8, SB = NTHREADS / TX;
  p.tiles_a = (p.L[p.a] + TX - 1) / TX;
  p.tiles_b = (p.L[p.b] + N * SB - 1) / (N * SB);
  p.nblocks = (long long)p.tiles_a * p.tiles_b * p.nbatch_total;
  if (p.nblocks <= 0) return hipSuccess;
  const dim3 grid((unsigned)p.nblocks), block(NTHREADS);
  const size_t l4 = side_lds<US, UD, 1, unsigned>(p), l8 = side_lds<US, UD, 1, i64>(p);
  if (p.below_4g && p.nontemporal) hipLaunchKernelGGL((reshape_rows<BYTES, US, UD, TX, unsigned, true>), grid, block, l4, s, p);
  else if (p.below_4g) hipLaunchKernelGGL((reshape_rows<BYTES, US, UD, TX, unsigned, false>), grid, block, l4, s, p);
  else if (p.nontemporal) hipLaunchKernelGGL((reshape_rows<BYTES, US, UD, TX, i64, true>), grid, block, l8, s, p);
  else hipLaunchKernelGGL((reshape_rows<BYTES, US, UD, TX, i64, false>), grid, block, l8, s, p);
  return hipGetLastError();
}

// Tile shapes (a x b x batch slices).
//   small   32 x 32 of 16 KiB: the least latency, and little lost where an
//           axis does not fill its tiles
//   large   16 elements a thread (8 of 16 bytes), rows of at least 256 bytes
//           on both sides: an element costs more instructions than bytes
//   narrow  16 wide, for an axis of at most 16 values (the phase order's
//           split axes), where a 32-wide tile stays half empty
// Measured us a pass (large / small / narrow; before there were several: 32 x
// 32 x 2, element addresses in 64 bits):
//   512^3 int64 chain, two hops               844 / 963; before 944
//   400 x 380 x 392 4-byte, permuted          179 / 294
//   352 x 416 x 256 int64 chain               332 / 360; 368
//   416 x 352 x 64 int64 chain (72 MB a side) 104 / 109; 117
//   384 x 64 x 224 int64 chain (42 MB)        70 / 57; 80
//   512 x 64 x 96 4-byte, permuted (12 MB)    26.5 / 18.8; 22.7
//   352 x 256 x 96 int64 chain, tiles 3/4 full 91.6 / 78.1; 87.2
//   512^3 phase order, complex float (calls)  5752 / 3160 / 3160; 5854
//   256^3 phase order, complex float          1110 / 519 / 463; 923
//   64^3 phase order, complex float           177 / 141 / 148; 179
// (the split axes of 512^3 are 16 x 32 points: a large tile is an eighth
// full; 215 x 13 x 310 16-byte, 14 MB, 21.2 us small, 19.4 narrow; calls of
// 512 x 30 x 30 in phase order, complex double, 7 MB, 193 and 179.)  Hence:
// where an axis is short the narrow tile, of fewer than 16 bytes from 128
// MiB over the element size on; the large one from 64 MiB a side on unless
// rounding the axes up to it moves a fifth more than rounding them up to the
// small one; else the small one.
struct TileForm {
  int a, b, n;
};
constexpr TileForm small_tile(int bytes) { return {32, 32, bytes > 8 ? 1 : 2}; }
constexpr TileForm large_tile(int bytes) {
  return bytes == 16 ? TileForm{64, 32, 1} : (bytes == 8 ? TileForm{64, 64, 1} : TileForm{128, 64, 1});
}
constexpr TileForm narrow_tile(int bytes, bool along_a) {
  return along_a ? TileForm{16, 32, bytes == 16 ? 2 : 4} : TileForm{32, 16, bytes == 16 ? 2 : 4};
}
// LDS of a tile: the elements and both sides' pair tables.
size_t tile_lds(const ReshapeLaunch &p, TileForm f) {
  const int pairs = (p.src.uniform ? 0 : p.ss.np[0] * p.ss.np[1]) + (p.dst.uniform ? 0 : p.sd.np[0] * p.sd.np[1]);
  return (size_t)f.n * f.a * (f.b + 1) * p.elem_bytes + (size_t)pairs * 3 * f.n * (p.below_4g ? 4 : 8);
}
TileForm tile_form(const ReshapeLaunch &p) {
  const int bytes = p.elem_bytes, la = p.L[p.a], lb = p.L[p.b];
  const TileForm small = small_tile(bytes);
  if (bytes == 12 || bytes == 24) return small;
  double side = bytes;
  for (int d = 0; d < p.ndim; d++) side *= p.L[d];
  auto rounded = [&](TileForm f) { return (double)((la + f.a - 1) / f.a * f.a) * ((lb + f.b - 1) / f.b * f.b); };
  const TileForm large = large_tile(bytes), narrow = narrow_tile(bytes, la <= 16);
  if (std::min(la, lb) <= 16 && (bytes == 16 || side > (double)(128 << 20) / bytes) && tile_lds(p, narrow) <= kTileLds)
    return narrow;
  if (side >= (64 << 20) && rounded(large) <= 1.25 * rounded(small)) return large;
  // (two slices' pair tables of 512 pairs a side in 64 bits: 66 KiB in all)
  return tile_lds(p, small) <= kTileLds ? small : large;
}

template <int BYTES, bool US, bool UD>
hipError_t launch_owned(ReshapeLaunch &p, hipStream_t s) {
  if (p.same_order) {
    if (p.L[p.a] <= 64) return launch_rows<BYTES, US, UD, 64>(p, s);
    return launch_rows<BYTES, US, UD, 256>(p, s);
  }
  const TileForm f = tile_form(p);
  if constexpr (BYTES != 12 && BYTES != 24) {
    constexpr TileForm large = large_tile(BYTES), na = narrow_tile(BYTES, true), nb = narrow_tile(BYTES, false);
    if (f.a == na.a) return launch_tile<BYTES, US, UD, na.a, na.b, na.n>(p, s);
    if (f.b == nb.b) return launch_tile<BYTES, US, UD, nb.a, nb.b, nb.n>(p, s);
    if (f.a == large.a) return launch_tile<BYTES, US, UD, large.a, large.b, large.n>(p, s);
  }
  constexpr TileForm small = small_tile(BYTES);
  return launch_tile<BYTES, US, UD, small.a, small.b, small.n>(p, s);
}

// ---- coordinates without an owner, or very many rank positions --------------

template <int BYTES, bool US, bool UD>
hipError_t launch_typed(ReshapeLaunch &p, hipStream_t s) {
  if (p.owned) return launch_owned<BYTES, US, UD>(p, s);
  if constexpr (BYTES == 12 || BYTES == 24) {
    return hipErrorInvalidValue;  // moved as words by the caller
  } else {
    if (p.a != p.b) {
      p.tiles_a = (p.L[p.a] + TILE - 1) / TILE;
      p.tiles_b = (p.L[p.b] + TILE - 1) / TILE;
      const int slices = tile_slices(p.elem_bytes);
      p.nblocks = (long long)p.tiles_a * p.tiles_b * ((p.nbatch_total + slices - 1) / slices);
    } else {
      p.tiles_a = (p.L[p.a] + NTHREADS * 4 - 1) / (NTHREADS * 4);
      p.tiles_b = 1;
      p.nblocks = (long long)p.tiles_a * p.nbatch_total;
    }
    if (p.nblocks <= 0) return hipSuccess;
    const dim3 grid((unsigned)p.nblocks), block(NTHREADS);
    auto launch = [&](auto nt) {
      constexpr bool NT = decltype(nt)::value;
      if (p.a != p.b) hipLaunchKernelGGL((reshape_tile2d<BYTES, US, UD, tile_slices(BYTES), NT>), grid, block, 0, s, p);
      else hipLaunchKernelGGL((reshape_run1d<BYTES, US, UD, NT>), grid, block, 0, s, p);
    };
    if (p.nontemporal) launch(std::true_type{});
    else launch(std::false_type{});
    return hipGetLastError();
  }
}

template <int BYTES>
hipError_t launch_bytes(ReshapeLaunch &p, hipStream_t s) {
  bool us = p.src.uniform, ud = p.dst.uniform;
  if (us && ud) return launch_typed<BYTES, true, true>(p, s);
  if (us) return launch_typed<BYTES, true, false>(p, s);
  if (ud) return launch_typed<BYTES, false, true>(p, s);
  return launch_typed<BYTES, false, false>(p, s);
}

}  // namespace

size_t reshape_tile_lds(const ReshapeLaunch &p) { return p.owned && !p.same_order ? tile_lds(p, tile_form(p)) : 0; }

// Tile counts and grid size are filled here so the host only chooses axes.
int launch_reshape(const ReshapeLaunch &p0, void *stream) {
  ReshapeLaunch p = p0;
  hipStream_t s = (hipStream_t)stream;
  long long batch = 1;
  for (int k = 0; k < p.nbatch; k++) batch *= p.L[p.batch_axis[k]];
  p.nbatch_total = batch;
  switch (p.elem_bytes) {
    case 1: return (int)launch_bytes<1>(p, s);
    case 2: return (int)launch_bytes<2>(p, s);
    case 4: return (int)launch_bytes<4>(p, s);
    case 8: return (int)launch_bytes<8>(p, s);
    case 12: return (int)launch_bytes<12>(p, s);
    case 16: return (int)launch_bytes<16>(p, s);
    case 24: return (int)launch_bytes<24>(p, s);
    default: return (int)hipErrorInvalidValue;  // other sizes are split into words by the caller
  }
}

}  // namespace dm

// ---- plain copy, the calibration reference for bandwidth and counters ------
namespace dm {
namespace {
// One 16-byte element per thread, 4 KiB per workgroup, non-temporal: the
// fastest plain copy measured here (6.4 TB/s for 2 GiB; 16 KiB per
// workgroup without the hint: 5.6-5.8 TB/s).
__global__ __launch_bounds__(256) void copy16_kernel(const uint4 *__restrict__ src, uint4 *__restrict__ dst,
                                                     long long n) {
  typedef unsigned int v4 __attribute__((ext_vector_type(4)));
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) {
    const v4 v = __builtin_nontemporal_load(reinterpret_cast<const v4 *>(src) + i);
    __builtin_nontemporal_store(v, reinterpret_cast<v4 *>(dst) + i);
  }
}
}  // namespace

int launch_copy16(const void *src, void *dst, long long n16, void *stream) {
  long long blocks = (n16 + 255) / 256;
  if (blocks <= 0) return 0;
  hipLaunchKernelGGL(copy16_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     (const uint4 *)src, (uint4 *)dst, n16);
  return (int)hipGetLastError();
}
}  // namespace dm
