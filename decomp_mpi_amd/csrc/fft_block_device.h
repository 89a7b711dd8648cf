// One stage of a multi-dimensional LDS tile (fft_block.hip's tiles of
// distributed arrays, batch_planes.hip's planes of local ones): elements in
// one padded linear order, the transformed dimension at stride s in it.
#pragma once
#include "fft_device.h"

namespace dm {
namespace fftdev {

constexpr int kPer = 16;  // points per thread (of most tiles)
template <typename R, bool CT>
using lds_tw = __attribute__((address_space(3))) typename tw_local<R, CT>::type;

// Butterfly b of a stage: its first point's element index without the
// butterfly's place along the axis, and that place.
__device__ __forceinline__ void butterfly(const BlockStage &st, int b, int *base, int *j) {
  const int q = fdiv(b, st.m_s), inner = b - q * st.s;
  const int outer = fdiv(q, st.m_nr);
  *j = q - outer * st.nr;
  *base = outer * st.span + inner;
}

template <typename R, bool INV, int RADIX, int NTH, bool CT, int PER = kPer>
__device__ __forceinline__ void block_stage(cx<R> *buf, const BlockStage &st, int points, const lds_tw<R, CT> *tw) {
  constexpr int K = (PER + RADIX - 1) / RADIX;
  const int nb = points / RADIX;
  cx<R> v[K][RADIX];
  int dst[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int b = threadIdx.x + k * NTH;
    dst[k] = -1;
    if (b < nb) {
      int base, j;
      butterfly(st, b, &base, &j);
      const int jn = fdiv(j, st.m_ns), jj = j - jn * st.ns;
#pragma unroll
      for (int r = 0; r < RADIX; r++) v[k][r] = buf[lds_pad(base + (j + r * st.nr) * st.s)];
      if (st.ns > 1) {
        const lds_tw<R, CT> *t = tw + st.tw + jj;
#pragma unroll
        for (int r = 1; r < RADIX; r++) v[k][r] = twmul<INV, CT>(v[k][r], t, (r - 1) * st.ns);
      }
      dft<R, INV, RADIX>(v[k]);
      dst[k] = base + (jn * st.ns * RADIX + jj) * st.s;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K; k++)
    if (dst[k] >= 0)
#pragma unroll
      for (int r = 0; r < RADIX; r++) buf[lds_pad(dst[k] + r * st.ns * st.s)] = v[k][r];
  __syncthreads();
}

}  // namespace fftdev
}  // namespace dm
