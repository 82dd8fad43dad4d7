// finalize.hpp -- adding up the partial sums of a split pair sum.
//
// A small sum is split over sources into many partials (54-80 at 7,682 targets) so
// that its waves fill the chip.  With a thread per target they were then added one
// after the other by 121 waves that wait on every load: 27 us behind a 37 us sum.
// From kFinSplits on, W waves share 64 targets: wave w adds splits w, w + W, ... with
// four splits' loads in flight, and the W sums are added in order through LDS:
// 5 us.  Below it one thread a target is as fast and needs no LDS.
#pragma once

#include <hip/hip_runtime.h>

#include "lpm_internal.hpp"

namespace lpm {

constexpr int kFinSplits = 16;
constexpr int kFinWays = 8;
constexpr int fin_threads(int w) { return w == 1 ? 256 : 64 * w; }

// A = the sum over the splits of target record i's NO partials.  False for a
// thread with nothing to store.
template <int NO, int W>
__device__ __forceinline__ bool sum_partials(const FinArgs& f, int& i, double (&A)[NO]) {
  const int way = W == 1 ? 0 : threadIdx.x >> 6;
  i = W == 1 ? blockIdx.x * 256 + threadIdx.x : blockIdx.x * 64 + (threadIdx.x & 63);
#pragma unroll
  for (int k = 0; k < NO; ++k) A[k] = 0.0;
  const size_t step = (size_t)NO * f.nt;
  if (i < f.nt) {
    const double* ps = f.partial + way * step + i;
    int s = way;
    for (; s + 3 * W < f.nsplit; s += 4 * W, ps += 4 * W * step) {
      double v[4][NO];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int k = 0; k < NO; ++k) v[e][k] = ps[e * W * step + (size_t)k * f.nt];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int k = 0; k < NO; ++k) A[k] += v[e][k];
    }
    for (; s < f.nsplit; s += W, ps += W * step)
#pragma unroll
      for (int k = 0; k < NO; ++k) A[k] += ps[(size_t)k * f.nt];
  }
  if constexpr (W > 1) {
    __shared__ double sh[W - 1][NO][64];
    if (way > 0)
#pragma unroll
      for (int k = 0; k < NO; ++k) sh[way - 1][k][threadIdx.x & 63] = A[k];
    __syncthreads();
    if (way > 0) return false;
#pragma unroll
    for (int w = 0; w < W - 1; ++w)
#pragma unroll
      for (int k = 0; k < NO; ++k) A[k] += sh[w][k][threadIdx.x];
  }
  return i < f.nt;
}

// Launch KERNEL<..., W>(f) with the way count for f's splits.
#define LPM_LAUNCH_FIN(f, st, KERNEL, ...)                                                                       \
  do {                                                                                                           \
    if ((f).nsplit >= ::lpm::kFinSplits)                                                                         \
      hipLaunchKernelGGL((KERNEL<__VA_ARGS__, ::lpm::kFinWays>), dim3(((f).nt + 63) / 64),                        \
                         dim3(::lpm::fin_threads(::lpm::kFinWays)), 0, st, f);                                   \
    else                                                                                                         \
      hipLaunchKernelGGL((KERNEL<__VA_ARGS__, 1>), dim3(((f).nt + 255) / 256), dim3(::lpm::fin_threads(1)), 0, st, \
                         f);                                                                                     \
  } while (0)

}  // namespace lpm
