// cull_kernels.hpp -- PSE and shallow-water sums that leave out the tiles whose
// kernel factor is exactly zero.
//
// Every PSE term carries exp(-q), q the squared separation over eps^2, and in the
// sum over all pairs nearly every term is zero: exp2(-q') is 0 in FP32 from q' = 150
// (10.2 eps), exp(-q) in FP64 from q = 746 (27.3 eps), and a finite value times 0
// adds nothing.  A source tile whose ball is farther than that from the ball of the
// wave's targets adds only zeros and is passed over; every other pair keeps the
// arithmetic of the all-pairs kernel.  At 512^2 with eps = 2 h the reach is 20 h:
// about 3,000 of 262,144 sources per target remain.
//
// A tile within reach may still leave the sums as they are: they are FP64, and adding
// a tile's partial p with |p| < 2^-54 |S| to a sum S rounds to S.  So the tiles near
// the targets come first, and each of the others is tested against the sums that it
// would be added to: its partials are at most
//   64 V (3/2) q^3 sqrt(q') exp(-q)   for q >= 16
// with V a bound of the tile's weights, q the squared distance of the balls over eps^2
// and q' the same in record units.  The sums are bit by bit those with the tile added.
// A sum that is zero or not finite (no near tile, exact cancellation) lets no tile be
// passed over.  The FP64 sphere gradient at level 6 took 12.2 ms over all tiles in
// reach and takes 1.9; PSE-8 at 512^2 in FP32 366 and 321 us.
//
// Layout: records in spatial order, one wave per 64 R targets, source tiles of 64
// records.  64 tiles are tested at once, one per lane; the ballot drives a scalar
// loop over the tiles that remain, whose records are read with scalar loads.  Splits
// take every nsplit-th tile, so that they share each neighbourhood evenly.
#pragma once

#include "tiles.hpp"

namespace lpm {

constexpr int CULL_TILE = 64;
constexpr float CULL_Q32 = 150.f;   // exp2(-q) rounds to 0 (2^-150 is half the least denormal)
constexpr double CULL_Q64 = 746.0;  // exp(-q) rounds to 0 (ln of half the least denormal: -745.2)

struct CullArgs {
  const void* tgt;
  const void* src;
  double* partial;        // [nsplit][NOUT][nt]
  const float4* tballs;   // per wave
  const float4* sballs;   // per CULL_TILE sources
  const int* tgt_order;   // particle of every target record, null where no pair is a self pair
  int nt, ns, nsplit, n_wtiles, n_stiles;
  float reach;            // separation in record units beyond which terms are zero
  // shallow water: balls per FAR_TILE; the tiles that are far of each other are not
  // this kernel's (null: all are)
  const float4* far_tballs = nullptr;
  const float4* far_sballs = nullptr;
  // exponents of the tiles' weights (see BallSet::mag), null: every tile in reach is
  // added.  Weights of a term: w0 + value w1 (Laplacian, interpolation), or w0 max(1, w1)
  const float2* tmag = nullptr;
  const float2* smag = nullptr;
  int product = 0;
  float near_reach = 0.f;  // separation up to which tiles come first
  const float4* gballs = nullptr;  // per 64 source tiles; null: every group's tiles are looked at
};

// A tile's partials stay below 2^e: e from the exponent of its weights and the squared
// separation in record units (FP32: q log2 e).
template <typename T>
__device__ __forceinline__ float tile_exponent(float weights, float q) {
  constexpr float kLog2E = sizeof(T) == 4 ? 1.f : 1.442695f;
  return weights + 9.f + 3.5f * __builtin_amdgcn_logf(q) - kLog2E * 0.9999f * q;
}

// The sums of one source tile, records [j0, j1), for the wave's targets.
template <class P, typename T, int R, bool SELF>
__device__ __forceinline__ void cull_tile(const Vec4<T> t[R], const int tid[R], const T* __restrict__ src, int j0,
                                          int j1, double S[R][P::NOUT]) {
  constexpr int NO = P::NOUT;
  T p[R][NO];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int k = 0; k < NO; ++k) p[r][k] = (T)0;
  T sv[P::NW];
#pragma unroll
  for (int q = 0; q < P::NW; ++q) sv[q] = src[(size_t)j0 * P::NW + q];
#pragma unroll 2
  for (int j = j0; j < j1; ++j) {
    const int jn = j + 1 < j1 ? j + 1 : j;
    T sn[P::NW];
#pragma unroll
    for (int q = 0; q < P::NW; ++q) sn[q] = src[(size_t)jn * P::NW + q];
    W4<T> w[R];
    T f[R];
#pragma unroll
    for (int r = 0; r < R; ++r) P::arg(t[r], sv, w[r]);
#pragma unroll
    for (int r = 0; r < R; ++r) f[r] = P::trans(w[r]);
    bool mine = false;
    if constexpr (SELF) {
      const int sidx = rec_index(sv, P::IDX);
#pragma unroll
      for (int r = 0; r < R; ++r) mine = mine || sidx == tid[r];
    }
    if (SELF && __any(mine)) {  // one source in every few hundred
      const int sidx = rec_index(sv, P::IDX);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        T tmp[NO];
#pragma unroll
        for (int k = 0; k < NO; ++k) tmp[k] = (T)0;
        P::acc(sv, w[r], f[r], tmp);
#pragma unroll
        for (int k = 0; k < NO; ++k) p[r][k] += sidx == tid[r] ? (T)0 : tmp[k];
      }
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) P::acc(sv, w[r], f[r], p[r]);
    }
#pragma unroll
    for (int q = 0; q < P::NW; ++q) sv[q] = sn[q];
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int k = 0; k < NO; ++k) S[r][k] += (double)p[r][k];
}

// FAR: the policy of the tiles beyond reach, void to pass over them.
template <class P, class FAR, typename T, int R>
static __global__ __launch_bounds__(256) void cull_sum_kernel(const void* __restrict__ tgt,
                                                              const void* __restrict__ srcv,
                                                              double* __restrict__ partial, CullArgs a) {
  fill_tables<P::TABLE>();
  constexpr int NO = P::NOUT;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nblk_t = (a.n_wtiles + 3) >> 2;
  const int split = blockIdx.x / nblk_t;
  const int wtile = __builtin_amdgcn_readfirstlane((blockIdx.x - split * nblk_t) * 4 + wid);
  if (wtile >= a.n_wtiles) return;  // wave-uniform
  const Vec4<T>* tg = reinterpret_cast<const Vec4<T>*>(tgt);
  const T* src = reinterpret_cast<const T*>(srcv);
  Vec4<T> t[R];
  int tid[R];
  double S[R][NO];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = min(wtile * 64 * R + r * 64 + lane, a.nt - 1);
    t[r] = tg[i];
    tid[r] = a.tgt_order ? a.tgt_order[i] : -1;
#pragma unroll
    for (int k = 0; k < NO; ++k) S[r][k] = 0.0;
  }
  const float4 tb = a.tballs[wtile];
  const bool test = __is_same(FAR, void) && a.smag;
  auto run = [&](int tile, bool touch, bool near) {
    const int j0 = tile * CULL_TILE, j1 = min(a.ns, j0 + CULL_TILE);
    if (touch)
      cull_tile<P, T, R, true>(t, tid, src, j0, j1, S);
    else if (__is_same(FAR, void) || near)
      cull_tile<P, T, R, false>(t, tid, src, j0, j1, S);
    else if constexpr (!__is_same(FAR, void))
      cull_tile<FAR, T, R, false>(t, tid, src, j0, j1, S);
  };
  unsigned long long later = 0;  // of the first 64 groups of 64 tiles: holds tested tiles
  unsigned long long groups = ~0ull;  // of 64 groups: within reach
  for (int base = 0; base < a.n_stiles; base += 64) {
    if constexpr (__is_same(FAR, void)) {
      if (a.gballs) {
        if ((base & 4095) == 0) {
          const int g = (base >> 6) + lane;
          bool in = false;
          if (g * 64 < a.n_stiles) {
            const float4 gb = a.gballs[g];
            const float th = 1.0001f * (a.reach + tb.w + gb.w);
            in = !(ball_d2(tb, gb) > th * th);
          }
          groups = __ballot(in);
        }
        if (!((groups >> ((base >> 6) & 63)) & 1)) continue;
      }
    }
    const int mine = base + lane;
    bool near = false, touch = false, own = false, first = true;
    if (mine < a.n_stiles) {
      const float4 sb = a.sballs[mine];
      const float d2 = ball_d2(tb, sb);
      const float th = 1.0001f * (a.reach + tb.w + sb.w);
      near = !(d2 > th * th);
      touch = a.tgt_order && balls_touch(d2, tb, sb);
      own = (mine & (a.nsplit - 1)) == split;
      if constexpr (!__is_same(FAR, void)) {
        constexpr int W = FAR_TILE / (64 * R), B = FAR_TILE / CULL_TILE;
        if (a.far_tballs) own = own && !tiles_far_swe(a.far_tballs[wtile / W], a.far_sballs[mine / B], a.reach);
      }
      if (test) {
        const float th1 = 1.0001f * (a.near_reach + tb.w + sb.w);
        first = !(d2 > th1 * th1);
      }
    }
    const unsigned long long m_near = __ballot(near), m_touch = __ballot(touch);
    unsigned long long todo = __ballot(own);
    if constexpr (__is_same(FAR, void)) todo &= m_near;
    if (test) {
      const unsigned long long m_first = __ballot(first);
      if (base < 4096 && (todo & ~m_first)) later |= 1ull << (base >> 6);
      todo &= m_first;
    }
    while (todo) {
      const int b = __builtin_ctzll(todo);
      todo &= todo - 1;
      run(base + b, (m_touch >> b) & 1, (m_near >> b) & 1);
    }
  }
  if constexpr (__is_same(FAR, void)) {
    if (test) {
      // exponent below which a partial changes none of the wave's sums
      auto floor_exponent = [&]() {
        float e = __builtin_huge_valf();
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int k = 0; k < NO; ++k) {
            const double v = S[r][k];
            const float ev = v != 0.0 && __builtin_isfinite(v) ? (float)(__builtin_amdgcn_frexp_exp(v) - 1)
                                                               : -__builtin_huge_valf();
            e = fminf(e, ev);
          }
        for (int m = 32; m > 0; m >>= 1) e = fminf(e, __shfl_xor(e, m));
        return e - 55.f;
      };
      float floor_e = floor_exponent();
      const float value = a.tmag[wtile].x;
      for (int base = 0; base < a.n_stiles; base += 64) {
        if (base < 4096 && !((later >> (base >> 6)) & 1)) continue;
        const int mine = base + lane;
        bool cand = false;
        float most = 0.f;
        if (mine < a.n_stiles && (mine & (a.nsplit - 1)) == split) {
          const float4 sb = a.sballs[mine];
          const float d2 = ball_d2(tb, sb);
          const float th = 1.0001f * (a.reach + tb.w + sb.w), th1 = 1.0001f * (a.near_reach + tb.w + sb.w);
          cand = !(d2 > th * th) && d2 > th1 * th1;
          const float2 w = a.smag[mine];
          const float gap = 0.9999f * sqrtf(d2) - tb.w - sb.w;
          most = tile_exponent<T>(a.product ? w.x + fmaxf(w.y, 0.f) : fmaxf(w.x, value + w.y) + 1.f, gap * gap);
        }
        unsigned long long todo;
        while ((todo = __ballot(cand && !(most < floor_e)))) {
          const int b = __builtin_ctzll(todo);
          run(base + b, false, true);
          if (lane == b) cand = false;
          floor_e = floor_exponent();
        }
      }
    }
  }
  double* out = partial + (size_t)split * NO * a.nt;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = wtile * 64 * R + r * 64 + lane;
    if (i < a.nt) {
#pragma unroll
      for (int k = 0; k < NO; ++k) out[(size_t)k * a.nt + i] = S[r][k];
    }
  }
}

using CullFn = void (*)(const void*, const void*, double*, CullArgs);

}  // namespace lpm
