// tiles.hpp -- bounding balls of tiles of consecutive records.
//
// The tile paths (far_kernels.hpp, cull_kernels.hpp) choose a tile's treatment from
// two balls, one around its sources and one around a wave's or block's targets.
// With the records in spatial order (lpm_order.hip) the balls are small.
#pragma once

#include "pair_kernels.hpp"

namespace lpm {

// One set of records: n records of `words` values, `tile` records to a ball (at most
// 256), coordinates in the first `dims` words.  A ball is {centre, radius}; its radius
// is infinite when any word of `finite_mask` is not finite, so that the tile gets no
// shortcut and its infinities and NaN spread as in the sum over all pairs.
template <typename T>
struct BallSet {
  const T* rec = nullptr;
  float4* out = nullptr;
  int words = 0, n = 0, tile = 64, dims = 2;
  unsigned finite_mask = 0;
  const int2* desc = nullptr;  // when set: (first record, count) of every ball
  int balls = 0;
};

template <typename T>
__device__ __forceinline__ void ball_of(const BallSet<T>& a, int b) {
  const int lane = threadIdx.x & 63;
  const int first = a.desc ? a.desc[b].x : b * a.tile;
  const int count = a.desc ? a.desc[b].y : min(a.tile, a.n - first);
  T c[4][3];
  bool bad = false;
  T lo[3] = {(T)3e38, (T)3e38, (T)3e38}, hi[3] = {(T)-3e38, (T)-3e38, (T)-3e38};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int i = q * 64 + lane;
#pragma unroll
    for (int k = 0; k < 3; ++k) c[q][k] = (T)0;
    if (i < count) {
      const T* r = a.rec + (size_t)(first + i) * a.words;
      for (int k = 0; k < a.words; ++k)
        if ((a.finite_mask >> k) & 1u) bad = bad || !isfinite(r[k]);
      for (int k = 0; k < a.dims; ++k) c[q][k] = r[k];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        lo[k] = fmin(lo[k], c[q][k]);
        hi[k] = fmax(hi[k], c[q][k]);
      }
    }
  }
  float mid[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) {
      lo[k] = fmin(lo[k], __shfl_xor(lo[k], m));
      hi[k] = fmax(hi[k], __shfl_xor(hi[k], m));
    }
    mid[k] = (float)(lo[k] + (T)0.5 * (hi[k] - lo[k]));
  }
  T d2 = (T)0;  // about the rounded centre
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (q * 64 + lane < count) {
      const T dx = c[q][0] - (T)mid[0], dy = c[q][1] - (T)mid[1], dz = c[q][2] - (T)mid[2];
      d2 = fmax(d2, dx * dx + dy * dy + dz * dz);
    }
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) d2 = fmax(d2, __shfl_xor(d2, m));
  bad = __any(bad) || count <= 0;
  if (lane == 0) {
    const float rad = bad ? __builtin_huge_valf() : (float)sqrt(d2) * 1.000001f;
    a.out[b] = make_float4(mid[0], mid[1], mid[2], rad);
  }
}

// One wave per ball, targets first.
template <typename T>
static __global__ __launch_bounds__(256) void tile_balls(BallSet<T> tgt, BallSet<T> src) {
  const int b = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (b < tgt.balls)
    ball_of(tgt, b);
  else if (b - tgt.balls < src.balls)
    ball_of(src, b - tgt.balls);
}

// Separation of two balls: squared centre distance.
__device__ __forceinline__ float ball_d2(const float4& a, const float4& b) {
  const float dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
  return dx * dx + dy * dy + dz * dz;
}
// Whether a point may lie in both balls (for any rounding; true for infinite radii):
// only then can the tile hold a target's own particle.
__device__ __forceinline__ bool balls_touch(float d2, const float4& a, const float4& b) {
  const float th = 1.001f * (a.w + b.w);
  return !(d2 > th * th);
}

constexpr int FAR_TILE = 256;     // sources per tile, targets per block of the far path

// Well separated: every target-source distance is at least the radius of the target
// block (|Y| >= 2 rho_t).  The norms and products above are then at most 9 times the
// denominator for the closest pairs and about equal to it for nearly all; errors
// against FP64 are the same with 3 rho_t, and fewer tiles go the VALU way.  The
// margins keep a pair of equal points (a self pair) out for any rounding of centres
// and radii; the lower bound keeps the split's low parts normal.
__device__ __forceinline__ bool tiles_far(const float4& t, const float4& s) {
  const float d2 = ball_d2(t, s);
  const float th = 1.001f * s.w + 2.002f * t.w;
  return d2 > th * th && d2 > 1e-28f;
}

// f^2 stays a normal number: pair distances are at least 1e-3 of the centres'
__device__ __forceinline__ bool tiles_far_swe(const float4& t, const float4& s, float reach) {
  const float d2 = ball_d2(t, s);
  const float th = 1.0001f * (reach + t.w + s.w);
  return tiles_far(t, s) && d2 > th * th && d2 > 1e-12f && d2 < 1e16f;
}

}  // namespace lpm
