// K5: several whole axes of a (virtually) distributed array in one pass.
//
// A tile holds every point of two or three axes (16 x 16 x 16 or 64 x 64
// complex doubles, twice that of complex floats) times T lines of one more
// axis, so those axes cost one read and one write of the array instead of
// one per axis.  The stage passes of the phase order (B_d- and A_d-point
// sub-axes) and the fused program of small arrays run this way.  512^3
// complex double, default split, phase order: FFT_1 2.44 -> 1.69 ms a forward
// (two passes for three), FFT_2 2.75 -> 0.81 ms (one for three: 4 GiB at
// 5.3 TB/s).
//
// The tile is one padded LDS array over its dimensions, innermost the one
// that is contiguous in memory.  A stage along a dimension of stride s takes
// butterflies whose lanes run along the dimensions inside it (s > 1), or
// along the butterflies themselves (s = 1); stages of different axes
// commute, so the host puts stages of an outer axis first and last, where
// they are fused with the load and the store and their lanes walk
// contiguous memory.  16 points per thread: a 16-point axis is one butterfly
// in registers, and 64 KiB of a tile are in flight from 256 threads.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fft_block_device.h"
#include "kernels.h"

namespace dm {
namespace {

using namespace fftdev;

constexpr int kThreadsD = 256;  // 4096 complex doubles
constexpr int kThreadsF = 512;  // 8192 complex floats

typedef __attribute__((address_space(3))) i64 lds_i64;

// Coordinates of tile element e, innermost dimension first.
__device__ __forceinline__ void decode(const FftBlock &p, int e, int *x) {
#pragma unroll
  for (int d = 0; d < DM_BLOCK_DIMS - 1; d++) {
    if (d < p.ndim - 1) {
      const int q = fdiv(e, p.dim[d].m_n);
      x[d] = e - q * p.dim[d].n;
      e = q;
    } else {
      x[d] = d == p.ndim - 1 ? e : 0;
      e = 0;
    }
  }
  x[DM_BLOCK_DIMS - 1] = p.ndim == DM_BLOCK_DIMS ? e : 0;
}

// Element offset of tile element e on one side (off: the side's tables of
// all dimensions, the lines' bases among them); *line: its line.
__device__ __forceinline__ i64 offset_of(const FftBlock &p, const lds_i64 *off, int e, int *line) {
  int x[DM_BLOCK_DIMS];
  decode(p, e, x);
  i64 a = 0;
  *line = 0;
#pragma unroll
  for (int d = 0; d < DM_BLOCK_DIMS; d++)
    if (d < p.ndim) {
      a += off[p.dim[d].at + x[d]];
      if (d == p.line_dim) *line = x[d];
    }
  return a;
}

// First stage on the loaded values (no stage twiddle; wl: the factors of a
// split axis's second half, or null).
template <typename R, bool INV, int RADIX, int NTH, bool CT>
__device__ __forceinline__ void block_load(cx<R> *buf, const FftBlock &p, const lds_i64 *off,
                                           const lds_tw<R, CT> *wl, int nl) {
  constexpr int K = kPer / RADIX;
  const BlockStage &st = p.st[0];
  const int nb = p.points / RADIX;
  const lds_i64 *along = off + p.dim[st.dim].at;
  const cx<R> *in = reinterpret_cast<const cx<R> *>(p.in);
  i64 a[K][RADIX];
  int base[K], j[K];
  bool ok[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int b = min((int)threadIdx.x + k * NTH, nb - 1);
    butterfly(st, b, &base[k], &j[k]);
    int line;
    const i64 o = offset_of(p, off, base[k], &line);  // at point 0 along the axis
    ok[k] = (int)threadIdx.x + k * NTH < nb && line < nl;
#pragma unroll
    for (int r = 0; r < RADIX; r++) a[k][r] = o - along[0] + along[j[k] + r * st.nr];
  }
  cx<R> v[K][RADIX];
  gather<K * RADIX>(&v[0][0], in, &a[0][0], p.stream_in);
#pragma unroll
  for (int k = 0; k < K; k++) {
    if ((int)threadIdx.x + k * NTH < nb) {
      if (!ok[k])
#pragma unroll
        for (int r = 0; r < RADIX; r++) v[k][r] = {0, 0};
      if (p.wtab != nullptr)
#pragma unroll
        for (int r = 0; r < RADIX; r++) v[k][r] = twmul<INV, CT>(v[k][r], wl, j[k] + r * st.nr);
      dft<R, INV, RADIX>(v[k]);
#pragma unroll
      for (int r = 0; r < RADIX; r++) buf[lds_pad(base[k] + (j[k] * RADIX + r) * st.s)] = v[k][r];
    }
  }
}

// Last stage of its axis (earlier points ns = nr), straight to memory.
template <typename R, bool INV, int RADIX, int NTH, bool CT>
__device__ __forceinline__ void block_store(const cx<R> *buf, const FftBlock &p, const lds_i64 *off,
                                            const lds_tw<R, CT> *tw, int nl) {
  constexpr int K = kPer / RADIX;
  const BlockStage &st = p.st[p.nstage - 1];
  const int nb = p.points / RADIX;
  const lds_i64 *along = off + p.dim[st.dim].at;
  cx<R> *out = reinterpret_cast<cx<R> *>(p.out);
  cx<R> v[K][RADIX];
  i64 a[K][RADIX];
  bool ok[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int b = min((int)threadIdx.x + k * NTH, nb - 1);
    int base, j, line;
    butterfly(st, b, &base, &j);
    const i64 o = offset_of(p, off, base, &line);
    ok[k] = (int)threadIdx.x + k * NTH < nb && line < nl;
#pragma unroll
    for (int r = 0; r < RADIX; r++) {
      v[k][r] = buf[lds_pad(base + (j + r * st.nr) * st.s)];
      a[k][r] = o - along[0] + along[j + r * st.nr];
    }
    if (st.ns > 1)
#pragma unroll
      for (int r = 1; r < RADIX; r++) v[k][r] = twmul<INV, CT>(v[k][r], tw + st.tw + j, (r - 1) * st.ns);
    dft<R, INV, RADIX>(v[k]);
  }
  scatter<K * RADIX, RADIX>(out, &a[0][0], &v[0][0], ok, p.stream_out);
}

// MX: schedules with radix 3, 5 or 7.  Two workgroups per CU by LDS.
template <typename R, bool INV, bool MX, bool CT>
__global__ __launch_bounds__(sizeof(R) == 8 ? kThreadsD : kThreadsF, sizeof(R) == 8 ? 2 : 4) void fft_block_kernel(FftBlock p) {
  constexpr int NTH = sizeof(R) == 8 ? kThreadsD : kThreadsF;
  typedef typename tw_local<R, CT>::type TwL;
  typedef typename tw_global<R>::type TwG;
  extern __shared__ __align__(16) char smem[];
  cx<R> *buf = reinterpret_cast<cx<R> *>(smem);
  char *at = smem + p.lds_tab;
  lds_i64 *in_off = (lds_i64 *)(at), *out_off = in_off + p.ntab;
  TwL *twl = reinterpret_cast<TwL *>(smem + p.lds_tw);
  const long long tile = blockIdx.x;
  const int T = p.line_dim >= 0 ? p.dim[p.line_dim].n : 1;
  const int nl = p.line_dim >= 0 ? min(T, p.lines - (int)(tile % p.tiles_u) * T) : 1;
  // both sides' offset tables (the lines' bases of this tile in their
  // dimension's place) and the twiddles
  const TwG *twg = reinterpret_cast<const TwG *>(p.twiddle);
  auto put = [&](int i, TwG w) {
    if constexpr (sizeof(TwL) == sizeof(TwG)) twl[i] = w;
    else twl[i] = TwL{w.x, w.y};
  };
  // (every table's first loads go out together)
  TwG tw0 = twg[min((int)threadIdx.x, p.ntw - 1)], w0{};
  const TwG *wtab = reinterpret_cast<const TwG *>(p.wtab);
  const int q = wtab != nullptr ? (int)(tile / p.tiles_u / p.wdiv % p.wlen) : 0;
  if (wtab != nullptr) w0 = wtab[min((int)threadIdx.x, p.wn - 1) * q];
  const int line_at = p.line_dim >= 0 ? p.dim[p.line_dim].at : p.ntab - 1;
  for (int i = threadIdx.x; i < p.ntab; i += NTH) {
    const bool l = i >= line_at && i < line_at + T;
    in_off[i] = l ? p.base_in[tile * T + (i - line_at)] : p.off_in[i];
    out_off[i] = l ? p.base_out[tile * T + (i - line_at)] : p.off_out[i];
  }
  if ((int)threadIdx.x < p.ntw) put(threadIdx.x, tw0);
  for (int i = threadIdx.x + NTH; i < p.ntw; i += NTH) put(i, twg[i]);
  if (wtab != nullptr) {
    if ((int)threadIdx.x < p.wn) put(p.ntw + threadIdx.x, w0);
    for (int x = threadIdx.x + NTH; x < p.wn; x += NTH) put(p.ntw + x, wtab[x * q]);
  }
  __syncthreads();
  const lds_tw<R, CT> *tw = (const lds_tw<R, CT> *)twl;
  int s0 = 0;
  const int s1 = p.fuse_out ? p.nstage - 1 : p.nstage;
  if (p.fuse_in) {
    switch (p.st[0].radix) {
      case 2: block_load<R, INV, 2, NTH, CT>(buf, p, in_off, tw + p.ntw, nl); break;
      case 4: block_load<R, INV, 4, NTH, CT>(buf, p, in_off, tw + p.ntw, nl); break;
      case 8: block_load<R, INV, 8, NTH, CT>(buf, p, in_off, tw + p.ntw, nl); break;
      case 16: block_load<R, INV, 16, NTH, CT>(buf, p, in_off, tw + p.ntw, nl); break;
      default: break;
    }
    s0 = 1;
  } else {
    i64 a[kPer];
    bool ok[kPer];
#pragma unroll
    for (int k = 0; k < kPer; k++) {
      const int e = threadIdx.x + k * NTH;
      int line;
      a[k] = offset_of(p, in_off, min(e, p.points - 1), &line);
      ok[k] = e < p.points && line < nl;
    }
    cx<R> v[kPer];
    gather<kPer>(v, reinterpret_cast<const cx<R> *>(p.in), a, p.stream_in);
#pragma unroll
    for (int k = 0; k < kPer; k++) {
      const int e = threadIdx.x + k * NTH;
      if (e < p.points) buf[lds_pad(e)] = ok[k] ? v[k] : cx<R>{0, 0};
    }
  }
  __syncthreads();
  for (int s = s0; s < s1; s++) {
    const BlockStage &st = p.st[s];
    switch (st.radix) {
      case 2: block_stage<R, INV, 2, NTH, CT>(buf, st, p.points, tw); break;
      case 4: block_stage<R, INV, 4, NTH, CT>(buf, st, p.points, tw); break;
      case 8: block_stage<R, INV, 8, NTH, CT>(buf, st, p.points, tw); break;
      case 16: block_stage<R, INV, 16, NTH, CT>(buf, st, p.points, tw); break;
      case 3: if constexpr (MX) block_stage<R, INV, 3, NTH, CT>(buf, st, p.points, tw); break;
      case 5: if constexpr (MX) block_stage<R, INV, 5, NTH, CT>(buf, st, p.points, tw); break;
      case 7: if constexpr (MX) block_stage<R, INV, 7, NTH, CT>(buf, st, p.points, tw); break;
      default: break;
    }
  }
  if (p.fuse_out) {
    switch (p.st[p.nstage - 1].radix) {
      case 2: block_store<R, INV, 2, NTH, CT>(buf, p, out_off, tw, nl); break;
      case 4: block_store<R, INV, 4, NTH, CT>(buf, p, out_off, tw, nl); break;
      case 8: block_store<R, INV, 8, NTH, CT>(buf, p, out_off, tw, nl); break;
      case 16: block_store<R, INV, 16, NTH, CT>(buf, p, out_off, tw, nl); break;
      default: break;
    }
  } else {
    i64 a[kPer];
    bool ok[kPer];
    cx<R> v[kPer];
#pragma unroll
    for (int k = 0; k < kPer; k++) {
      const int e = threadIdx.x + k * NTH, ec = min(e, p.points - 1);
      int line;
      a[k] = offset_of(p, out_off, ec, &line);
      ok[k] = e < p.points && line < nl;
      v[k] = buf[lds_pad(ec)];
    }
    scatter<kPer, 1>(reinterpret_cast<cx<R> *>(p.out), a, v, ok, p.stream_out);
  }
}

template <typename R, bool INV, bool MX, bool CT>
hipError_t launch_typed(const FftBlock &p, hipStream_t s) {
  auto k = fft_block_kernel<R, INV, MX, CT>;
  // once per kernel (a thread-safe static)
  static const hipError_t attr =
      hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL(k, dim3((unsigned)p.tiles), dim3(sizeof(R) == 8 ? kThreadsD : kThreadsF), p.lds, s, p);
  return hipGetLastError();
}

template <typename R, bool CT>
hipError_t launch_forms(const FftBlock &p, bool mx, hipStream_t s) {
  if (p.inverse) return mx ? launch_typed<R, true, true, CT>(p, s) : launch_typed<R, true, false, CT>(p, s);
  return mx ? launch_typed<R, false, true, CT>(p, s) : launch_typed<R, false, false, CT>(p, s);
}

}  // namespace

int fft_block_capacity(int dbl) { return kPer * (dbl ? kThreadsD : kThreadsF); }

void fft_block_lds(FftBlock *p) {
  const size_t es = p->dbl ? 16 : 8;
  auto up = [](size_t x) { return (x + 15) & ~(size_t)15; };
  size_t b = up((size_t)(lds_pad(p->points - 1) + 1) * es);
  p->lds_tab = (int)b;
  b += up((size_t)p->ntab * 2 * sizeof(i64));
  p->lds_tw = (int)b;
  b += (size_t)(p->ntw + p->wn) * (p->dbl || p->ctw ? 16 : 8);
  p->lds = b;
}

int launch_fft_block(const FftBlock &p, void *stream) {
  if (p.tiles <= 0) return 0;
  if (p.tiles >= (1LL << 31) || p.points > fft_block_capacity(p.dbl) || p.lds > 160 * 1024)
    return (int)hipErrorInvalidValue;
  bool mx = false;
  for (int i = 0; i < p.nstage; i++) mx = mx || (p.st[i].radix & (p.st[i].radix - 1)) != 0;
  hipStream_t s = (hipStream_t)stream;
  if (p.dbl) return (int)launch_forms<double, false>(p, mx, s);
  return (int)(p.ctw ? launch_forms<float, true>(p, mx, s) : launch_forms<float, false>(p, mx, s));
}

}  // namespace dm
