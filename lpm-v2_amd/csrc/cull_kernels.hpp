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
};

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
  for (int base = 0; base < a.n_stiles; base += 64) {
    const int mine = base + lane;
    bool near = false, touch = false, own = false;
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
    }
    const unsigned long long m_near = __ballot(near), m_touch = __ballot(touch);
    unsigned long long todo = __ballot(own);
    if constexpr (__is_same(FAR, void)) todo &= m_near;
    while (todo) {
      const int b = __builtin_ctzll(todo);
      todo &= todo - 1;
      const int j0 = (base + b) * CULL_TILE, j1 = min(a.ns, j0 + CULL_TILE);
      if ((m_touch >> b) & 1)
        cull_tile<P, T, R, true>(t, tid, src, j0, j1, S);
      else if (__is_same(FAR, void) || ((m_near >> b) & 1))
        cull_tile<P, T, R, false>(t, tid, src, j0, j1, S);
      else if constexpr (!__is_same(FAR, void))
        cull_tile<FAR, T, R, false>(t, tid, src, j0, j1, S);
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
