// K3, plane tiles: the last two axes of many independent local FFTs in one
// pass (DM_BATCH_TILE_PLANES).
//
// A tile is one or more whole planes of one transform, contiguous in memory,
// so an element's offset is its index in the tile.  The columns' first stage
// runs on the loaded values and their last one before the store (lanes walk
// contiguous memory in both), the rows' stages between them in LDS: four LDS
// exchanges for a 64 x 64 plane.  512 threads: planes of up to 4096 points at
// 8 points per thread with butterflies of up to 8 (several small planes fill
// a tile), complex-float planes of up to 8192 at 16.  At 16 points per thread
// on 256 the small tile's odd radices ran one after another in too few waves:
// two complex-double 3D transforms of odd lengths 30 us a batch, 27 at 8, and
// 1126 and 1101 us for 153 of them.  As row stages, then column stages, then
// a store from LDS, one plane per workgroup, the planes of the 256-transform
// complex-float batch took 149 and 202 us (3.0 TB/s), 114 and 160 so (3.8),
// with the vector ALU 95% busy.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fft_block_device.h"
#include "kernels.h"

namespace dm {
namespace {

using namespace fftdev;

constexpr int NTH = 512;

template <typename R>
using gptr = __attribute__((address_space(1))) cx<R> *;  // global memory
typedef __attribute__((address_space(4))) const BatchPlane cplane;  // scalar loads

__device__ __forceinline__ BlockStage stage_of(const cplane &S, int i) {
  BlockStage st;
  st.m_s = S.st[i].m_s;
  st.m_nr = S.st[i].m_nr;
  st.m_ns = S.st[i].m_ns;
  st.dim = 0;
  st.radix = S.st[i].radix;
  st.s = S.st[i].s;
  st.span = S.st[i].span;
  st.nr = S.st[i].nr;
  st.ns = S.st[i].ns;
  st.tw = S.st[i].tw;
  return st;
}

template <typename R, bool INV, int RADIX, int PER>
__device__ __forceinline__ void plane_load(cx<R> *buf, const BlockStage &st, gptr<R> data, int points, int live) {
  constexpr int K = (PER + RADIX - 1) / RADIX;
  const int nb = points / RADIX;
  cx<R> v[K][RADIX];
  int e[K], j[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int b = threadIdx.x + k * NTH;
    butterfly(st, min(b, nb - 1), &e[k], &j[k]);
    // absent elements read the tile's first ones; they are never stored
    const int at = b < nb && e[k] < live ? e[k] + j[k] * st.s : 0;
    const int step = b < nb && e[k] < live ? st.nr * st.s : 0;
#pragma unroll
    for (int r = 0; r < RADIX; r++) v[k][r] = {data[at + r * step].x, data[at + r * step].y};
  }
#pragma unroll
  for (int k = 0; k < K; k++)
    if ((int)threadIdx.x + k * NTH < nb) {
      dft<R, INV, RADIX>(v[k]);
#pragma unroll
      for (int r = 0; r < RADIX; r++) buf[lds_pad(e[k] + (j[k] * RADIX + r) * st.s)] = v[k][r];
    }
}

template <typename R, bool INV, int RADIX, bool CT, int PER>
__device__ __forceinline__ void plane_store(const cx<R> *buf, const BlockStage &st, gptr<R> data, int points, int live,
                                            const lds_tw<R, CT> *tw) {
  constexpr int K = (PER + RADIX - 1) / RADIX;
  const int nb = points / RADIX;
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int b = threadIdx.x + k * NTH;
    int base, j;
    butterfly(st, min(b, nb - 1), &base, &j);
    cx<R> v[RADIX];
#pragma unroll
    for (int r = 0; r < RADIX; r++) v[r] = buf[lds_pad(base + (j + r * st.nr) * st.s)];
    if (st.ns > 1)
#pragma unroll
      for (int r = 1; r < RADIX; r++) v[r] = twmul<INV, CT>(v[r], tw + st.tw + j, (r - 1) * st.ns);
    dft<R, INV, RADIX>(v);
    if (b < nb && base < live)
#pragma unroll
      for (int r = 0; r < RADIX; r++) {
        const int at = base + (j + r * st.nr) * st.s;
        data[at].x = v[r].x;
        data[at].y = v[r].y;
      }
  }
}

// MX: schedules with odd radices.  Two workgroups per CU by LDS, three of
// complex-float planes of up to 4096 points.
template <typename R, bool INV, int PER, bool MX>
__global__ __launch_bounds__(NTH, 4) void batch_plane_kernel(BatchLaunch p) {
  constexpr bool CT = sizeof(R) == 4;  // compensated twiddle products
  typedef typename tw_local<R, CT>::type Tw;
  extern __shared__ __align__(16) char smem[];
  cx<R> *buf = reinterpret_cast<cx<R> *>(smem);
  Tw *twl = reinterpret_cast<Tw *>(smem + p.plane_tw);
  const lds_tw<R, CT> *tw = (const lds_tw<R, CT> *)twl;
  for (long long t = blockIdx.x; t < p.ntiles; t += gridDim.x) {
    const BatchTile d = p.tiles[t];
    const cplane &S = ((const cplane *)p.planes)[__builtin_amdgcn_readfirstlane(d.sched)];
    gptr<R> data = (gptr<R>)(p.data[d.xform]) + d.base;
    const int points = S.points, live = d.nl * S.plane, nst = S.nstage;
    const Tw *twg = reinterpret_cast<const Tw *>(p.twiddle) + S.tw_off;
    for (int i = threadIdx.x; i < S.ntw; i += NTH) twl[i] = twg[i];
    int s0 = 0;
    const int s1 = S.fuse_out ? nst - 1 : nst;
    if (S.fuse_in) {
      const BlockStage st = stage_of(S, 0);
      switch (st.radix) {
        case 2: plane_load<R, INV, 2, PER>(buf, st, data, points, live); break;
        case 4: plane_load<R, INV, 4, PER>(buf, st, data, points, live); break;
        case 8: plane_load<R, INV, 8, PER>(buf, st, data, points, live); break;
        case 16: if constexpr (PER == 16) plane_load<R, INV, 16, PER>(buf, st, data, points, live); break;
        default: break;
      }
      s0 = 1;
    } else {
      cx<R> v[PER];
#pragma unroll
      for (int k = 0; k < PER; k++) {
        const int e = threadIdx.x + k * NTH, at = e < live ? e : 0;
        v[k] = {data[at].x, data[at].y};
      }
#pragma unroll
      for (int k = 0; k < PER; k++) {
        const int e = threadIdx.x + k * NTH;
        if (e < points) buf[lds_pad(e)] = v[k];
      }
    }
    __syncthreads();
    for (int s = s0; s < s1; s++) {
      const BlockStage st = stage_of(S, s);
      switch (st.radix) {
        case 2: block_stage<R, INV, 2, NTH, CT, PER>(buf, st, points, tw); break;
        case 4: block_stage<R, INV, 4, NTH, CT, PER>(buf, st, points, tw); break;
        case 8: block_stage<R, INV, 8, NTH, CT, PER>(buf, st, points, tw); break;
        case 16: if constexpr (PER == 16) block_stage<R, INV, 16, NTH, CT, PER>(buf, st, points, tw); break;
        case 3: if constexpr (MX) block_stage<R, INV, 3, NTH, CT, PER>(buf, st, points, tw); break;
        case 5: if constexpr (MX) block_stage<R, INV, 5, NTH, CT, PER>(buf, st, points, tw); break;
        case 7: if constexpr (MX) block_stage<R, INV, 7, NTH, CT, PER>(buf, st, points, tw); break;
        case 11: if constexpr (MX) block_stage<R, INV, 11, NTH, CT, PER>(buf, st, points, tw); break;
        case 13: if constexpr (MX) block_stage<R, INV, 13, NTH, CT, PER>(buf, st, points, tw); break;
        default: break;
      }
    }
    if (S.fuse_out) {
      const BlockStage st = stage_of(S, nst - 1);
      switch (st.radix) {
        case 2: plane_store<R, INV, 2, CT, PER>(buf, st, data, points, live, tw); break;
        case 4: plane_store<R, INV, 4, CT, PER>(buf, st, data, points, live, tw); break;
        case 8: plane_store<R, INV, 8, CT, PER>(buf, st, data, points, live, tw); break;
        case 16: if constexpr (PER == 16) plane_store<R, INV, 16, CT, PER>(buf, st, data, points, live, tw); break;
        default: break;
      }
    } else {
#pragma unroll
      for (int k = 0; k < PER; k++) {
        const int e = threadIdx.x + k * NTH;
        if (e < live) {
          const cx<R> w = buf[lds_pad(e)];
          data[e].x = w.x;
          data[e].y = w.y;
        }
      }
    }
    __syncthreads();  // the next tile reuses the LDS tile
  }
}

template <typename R, bool INV, int PER, bool MX>
hipError_t launch_typed(const BatchLaunch &p, hipStream_t s) {
  auto k = batch_plane_kernel<R, INV, PER, MX>;
  // once per kernel (a thread-safe static)
  static const hipError_t attr =
      hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL(k, dim3((unsigned)p.grid), dim3(NTH), p.lds, s, p);
  return hipGetLastError();
}
template <typename R, int PER>
hipError_t launch_forms(const BatchLaunch &p, hipStream_t s) {
  if (p.primes)
    return p.inverse ? launch_typed<R, true, PER, true>(p, s) : launch_typed<R, false, PER, true>(p, s);
  return p.inverse ? launch_typed<R, true, PER, false>(p, s) : launch_typed<R, false, PER, false>(p, s);
}

constexpr int kSmall = 4096, kLarge = 8192;

}  // namespace

int batch_plane_capacity(int dbl) { return dbl ? kSmall : kLarge; }
int batch_plane_small() { return kSmall; }

size_t batch_plane_tw_at(int dbl, int points) {
  return ((size_t)(lds_pad(points - 1) + 1) * (dbl ? 16 : 8) + 15) & ~(size_t)15;
}

// Persistent grids: two workgroups per CU by registers, three of
// complex-float planes of up to 4096 points, fewer if LDS says so.
long long batch_plane_resident_groups(int dbl, int large, size_t lds) {
  int dev = 0, cus = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (cus <= 0) cus = 256;
  return (long long)cus * std::max(1, std::min(dbl || large ? 2 : 3, (int)((160 * 1024) / std::max<size_t>(lds, 1))));
}

int launch_batch_planes(const BatchLaunch &p, void *stream) {
  if (p.ntiles <= 0 || p.grid <= 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  if (p.plane == 1) return p.dbl ? (int)hipErrorInvalidValue : (int)launch_forms<float, 16>(p, s);
  return (int)(p.dbl ? launch_forms<double, 8>(p, s) : launch_forms<float, 8>(p, s));
}

}  // namespace dm
