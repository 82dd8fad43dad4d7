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
// is infinite when any word of `finite_mask` is not finite, or a coordinate beyond
// `limit`, so that the tile gets no shortcut and its infinities and NaN spread as in the
// sum over all pairs.
template <typename T>
struct BallSet {
  const T* rec = nullptr;
  float4* out = nullptr;
  int words = 0, n = 0, tile = 64, dims = 2;
  unsigned finite_mask = 0;
  float limit = __builtin_huge_valf();
  const int2* desc = nullptr;  // when set: (first record, count) of every ball
  int balls = 0;
  // when set: binary exponents e of the largest magnitudes among the words of each
  // mask, |word| < 2^e in the tile (-inf where all are zero)
  float2* mag = nullptr;
  unsigned mag_mask[2] = {0, 0};
};

// e with |v| < 2^e, -inf for 0 and +inf where v is not finite.
template <typename T>
__device__ __forceinline__ float exponent_above(T v) {
  if (v == (T)0) return -__builtin_huge_valf();
  return isfinite(v) ? (float)(ilogb(v) + 1) : __builtin_huge_valf();
}

template <typename T>
__device__ __forceinline__ void ball_of(const BallSet<T>& a, int b) {
  const int lane = threadIdx.x & 63;
  const int first = a.desc ? a.desc[b].x : b * a.tile;
  const int count = a.desc ? a.desc[b].y : min(a.tile, a.n - first);
  T c[4][3];
  bool bad = false;
  T big[2] = {(T)0, (T)0};
  T lo[3] = {(T)3e38, (T)3e38, (T)3e38}, hi[3] = {(T)-3e38, (T)-3e38, (T)-3e38};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int i = q * 64 + lane;
#pragma unroll
    for (int k = 0; k < 3; ++k) c[q][k] = (T)0;
    if (i < count) {
      const T* r = a.rec + (size_t)(first + i) * a.words;
      for (int k = 0; k < a.words; ++k)
      {
        if ((a.finite_mask >> k) & 1u) bad = bad || !isfinite(r[k]);
        if ((a.mag_mask[0] >> k) & 1u) big[0] = fmax(big[0], fabs(r[k]));
        if ((a.mag_mask[1] >> k) & 1u) big[1] = fmax(big[1], fabs(r[k]));
      }
      for (int k = 0; k < a.dims; ++k) {
        c[q][k] = r[k];
        bad = bad || fabs(r[k]) > (T)a.limit;
      }
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
  if (a.mag) {
#pragma unroll
    for (int m = 32; m > 0; m >>= 1)
#pragma unroll
      for (int q = 0; q < 2; ++q) big[q] = fmax(big[q], __shfl_xor(big[q], m));
    if (lane == 0) a.mag[b] = make_float2(exponent_above(big[0]), exponent_above(big[1]));
  }
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

// Balls around 64 balls each, one wave per group.
static __global__ __launch_bounds__(256) void group_balls(int n, const float4* __restrict__ balls,
                                                          float4* __restrict__ out) {
  const int g = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (g * 64 >= n) return;
  const float4 b = balls[min(g * 64 + lane, n - 1)];
  float lo[3] = {b.x, b.y, b.z}, hi[3] = {b.x, b.y, b.z};
  for (int m = 32; m > 0; m >>= 1)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      lo[k] = fminf(lo[k], __shfl_xor(lo[k], m));
      hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], m));
    }
  const float x = 0.5f * (lo[0] + hi[0]), y = 0.5f * (lo[1] + hi[1]), z = 0.5f * (lo[2] + hi[2]);
  const float dx = b.x - x, dy = b.y - y, dz = b.z - z;
  float rad = 1.000001f * (sqrtf(dx * dx + dy * dy + dz * dz) + b.w);
  if (!(rad < __builtin_huge_valf())) rad = __builtin_huge_valf();  // also where a centre is not a number
  for (int m = 32; m > 0; m >>= 1) rad = fmaxf(rad, __shfl_xor(rad, m));
  if (lane == 0) out[g] = make_float4(x, y, z, rad);
}

// Separation of two balls: squared centre distance.  Here and in the rules below no
// product is left for the compiler to fuse with a sum or not: the far and the cull
// kernel share out the tiles of a shallow-water sum by the same rule, each for itself,
// and with 1.001 s + 2.002 t fused one way in one and the other way in the other a tile
// pair on the line was summed twice or not at all.
__device__ __forceinline__ float ball_d2(const float4& a, const float4& b) {
  const float dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
  return fmaf(dz, dz, fmaf(dy, dy, dx * dx));
}
// Whether a point may lie in both balls (for any rounding; true for infinite radii):
// only then can the tile hold a target's own particle.
__device__ __forceinline__ bool balls_touch(float d2, const float4& a, const float4& b) {
  const float th = 1.001f * (a.w + b.w);
  return !(d2 > th * th);
}

constexpr int FAR_TILE = 256;     // sources per tile, targets per block of the far path
// Coordinates of far tiles: squared distances stay below 1.2e37, norms below 5e37.
constexpr float kFarLimit = 1e18f;

// Well separated: every target-source distance is at least the radius of the target
// block (|Y| >= 2 rho_t).  The norms and products above are then at most 9 times the
// denominator for the closest pairs and about equal to it for nearly all; errors
// against FP64 are the same with 3 rho_t, and fewer tiles go the VALU way.  The
// margins keep a pair of equal points (a self pair) out for any rounding of centres
// and radii; the lower bound keeps the split's low parts normal (kFarLimit: the norms finite).
__device__ __forceinline__ bool tiles_far(const float4& t, const float4& s) {
  const float d2 = ball_d2(t, s);
  const float th = fmaf(1.001f, s.w, 2.002f * t.w);
  return d2 > th * th && d2 > 1e-28f;
}

// Power of two about 1 / d, for the d2 of a far tile.
__device__ __forceinline__ float inverse_length(float d2) {
  const int e = ((int)(__float_as_uint(d2) >> 23) - 127) >> 1;
  return __uint_as_float((unsigned)(127 - e) << 23);
}

// f^2 stays a normal number: pair distances are at least 1e-3 of the centres'
__device__ __forceinline__ bool tiles_far_swe(const float4& t, const float4& s, float reach) {
  const float d2 = ball_d2(t, s);
  const float th = 1.0001f * (reach + t.w + s.w);
  return tiles_far(t, s) && d2 > th * th && d2 > 1e-12f && d2 < 1e16f;
}

}  // namespace lpm
