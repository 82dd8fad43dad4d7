// far_kernels.hpp -- the FP32 Biot-Savart, Green and shallow-water sums with the
// well-separated source tiles on the matrix units.
//
// The all-VALU pair (pair_kernels.hpp) is bound by VALU issue: 11-12 instructions,
// 31-36 cycles per 64 pairs and SIMD on MI355X.  Only the reciprocal (or log) has
// to run there.  For a block of targets and a tile of sources that are well
// separated, with X and Y the positions relative to the centre of the target block,
//   |x - y|^2 + e_x + e_y = (|X|^2 + e_x) + (|Y|^2 + e_y) - 2 X.Y
// loses nothing to cancellation, so it is a matrix product over 4 values, and the
// sum of s (x - y) is X (sum of s) - (sum of s Y), a matrix product as well:
//  * denominator: one v_mfma_f32_16x16x32_bf16 per 16 sources x 16 targets.  Every
//    FP32 value is split exactly into three bf16 values (8 significant bits each)
//    and the K = 32 slots hold 8 of the 9 partial products of each coordinate
//    (all but low x low, 2^-32 relative) and the two squared norms: an FP32
//    product at 16.7 cycles, where v_mfma_f32_16x16x4_f32 takes 32.5;
//  * rcp / log2 on the VALU, 8.2 cycles per 64 pairs, the floor of this form;
//  * accumulation (Biot-Savart): v_mfma_f32_4x4x1_16b_f32 with the source weights
//    (w Y, w) as its 4 rows, in FP32, 9.1 cycles per 64 pairs.  Its column layout
//    is the row layout of the first product, so nothing is moved between them.
//    Green sums have 1-2 outputs and accumulate with FMAs.
// Inner loop: 21.6 cycles per 64 pairs (4 column tiles; 30.6 when rcp and MFMA are
// interleaved by the scheduler, hence the scheduling barriers).
// Tiles that are not well separated, or hold a value that is not finite, take the
// VALU pair, self pairs included.  Records come in spatial order (lpm_order.hip).
#pragma once

#include "tiles.hpp"

namespace lpm {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int FAR_COLS = 4;       // 16-target column tiles per wave
constexpr int FAR_FOLD = 1024;    // sources per group, the unit of the source splits
constexpr int FAR_PART = 512;     // sources per FP32 partial sum (128 terms a lane)

// Exact split v = h + m + l into bf16 values, each in the high half of its word.
__device__ __forceinline__ void split3(float v, unsigned& h, unsigned& m, unsigned& l) {
  h = __float_as_uint(v) & 0xffff0000u;
  const float r = v - __uint_as_float(h);
  m = __float_as_uint(r) & 0xffff0000u;
  l = __float_as_uint(r - __uint_as_float(m)) & 0xffff0000u;
}
// low half of the result: high half of a; high half: high half of b
__device__ __forceinline__ unsigned pack_hi(unsigned a, unsigned b) { return (a >> 16) | b; }
constexpr unsigned kOneHi = 0x3f800000u;  // bf16 1.0 in the high half

// Source side (A operand) of one coordinate and of the norm; target side (B).
// Slots of a coordinate: hh, hm, mh, mm, hl, lh, ml, lm (source part first).
__device__ __forceinline__ u32x4 frag_src(float v) {
  unsigned h, m, l;
  split3(v, h, m, l);
  return u32x4{pack_hi(h, h), pack_hi(m, m), pack_hi(h, l), pack_hi(m, l)};
}
__device__ __forceinline__ u32x4 frag_src_norm(float n2) {
  unsigned h, m, l;
  split3(n2, h, m, l);
  // The bf16 MFMA truncates its sum to FP32: a mean error of -4.2e-8 of the
  // denominator, the same for every pair, where the VALU pair rounds to nearest.
  // 2^-24 of the source norm in one of the two free slots makes up for it: mean 1e-9
  // to 2e-8 and rms 5.0e-8, against an rms of 5.7e-8 of the VALU pair.
  const unsigned half_ulp = __float_as_uint(__uint_as_float(h) * 0x1p-24f) & 0xffff0000u;
  return u32x4{pack_hi(h, m), pack_hi(l, kOneHi), pack_hi(kOneHi, kOneHi), half_ulp >> 16};
}
__device__ __forceinline__ u32x4 frag_tgt(float v, bool norm) {
  unsigned h, m, l;
  split3(v, h, m, l);
  const u32x4 c{pack_hi(h, m), pack_hi(h, m), pack_hi(l, h), pack_hi(l, m)};
  const u32x4 n{pack_hi(kOneHi, kOneHi), pack_hi(kOneHi, h), pack_hi(m, l), kOneHi >> 16};
  return norm ? n : c;
}

// ----------------------------------------------------------- far policies
// DIMS coordinates; E: record word 3 holds e; W0 (and W1): weight words; NW weight
// sums accumulated by FMAs (0: by MFMA); trans: the VALU function; BLOCKS per CU.
template <bool USE_E>
struct FarSphereBS {
  using Near = SphereBS<float, USE_E>;
  static constexpr int DIMS = 3, W0 = 4, W1 = 4, NW = 0, BLOCKS = 4;
  static constexpr bool E = USE_E;
  __device__ __forceinline__ static float trans(float r2) { return fast_rcp(r2); }
};
struct FarPlaneBS {
  using Near = PlaneBS<float>;
  static constexpr int DIMS = 2, W0 = 2, W1 = 2, NW = 0, BLOCKS = 4;
  static constexpr bool E = false;
  __device__ __forceinline__ static float trans(float r2) { return fast_rcp(r2); }
};
template <bool USE_E>
struct FarSphereGreen {
  using Near = SphereGreen<float, USE_E>;
  static constexpr int DIMS = 3, W0 = 4, W1 = 5, NW = 2, BLOCKS = 4;
  static constexpr bool E = USE_E;
  __device__ __forceinline__ static float trans(float r2) { return fast_log2(r2); }
};
struct FarPlaneGreen {
  using Near = PlaneGreen<float>;
  static constexpr int DIMS = 2, W0 = 2, W1 = 2, NW = 1, BLOCKS = 4;
  static constexpr bool E = false;
  __device__ __forceinline__ static float trans(float r2) { return fast_log2(r2); }
};

// The shallow-water sums beyond the reach of the Laplacian's exponential, where only
// the vortex and divergence terms are left.  With z = X + i Y (target minus source),
// f = 1 / |z|^2 and c = vorticity + i divergence weight, the two velocity sums are
// those of c conj(z) f and the two gradient sums those of -c conj(z)^2 f^2; conj(z)
// is the difference of target and source, so both are matrix products of f and f^2
// with the source weights c, c conj(Z), c conj(Z)^2: three 4-row products, 42 cycles
// per 64 pairs against 66 on the VALU.  The other tiles are left to cull_sum_kernel,
// whose smaller tiles know the exponential's reach and which keeps more waves (sums
// of both: 301^2 3,480 -> 2,780 us, 512^2 26.1 -> 20.3 ms; with the near tiles in this
// kernel a reach over the whole domain cost 25 %).
struct FarSwePlane {
  using Near = SwePlane<float, true>;
  static constexpr int DIMS = 2, W0 = 2, W1 = 3, NW = 0, BLOCKS = 3;
  static constexpr bool E = false;
  __device__ __forceinline__ static float trans(float r2) { return fast_rcp(r2); }
};
template <class P>
inline constexpr bool kSwe = __is_same(P, FarSwePlane);

// LDS of one staged source tile: 16 steps of 16 sources, the MFMA A fragments
// (64 x 16 bytes a step) and the weights (16 x 16 bytes a step).
struct FarStage {
  u32x4 frag[16 * 64];
  f32x4 wgt[16 * 16];
};
struct FarStageSwe : FarStage {
  f32x4 wgt2[16 * 16];
};
template <class P>
struct FarStageOf {
  using T = FarStage;
};
template <>
struct FarStageOf<FarSwePlane> {
  using T = FarStageSwe;
};

// The direct VALU sum of one near tile for the wave's 64 targets (lane = target);
// SELF: the tile may hold the targets' own particles.  The near tiles are a tenth of
// the pairs at 1e10 and wait for their records more than for their arithmetic: with
// scalar loads 2, 4 and 6 sources ahead the velocity at level 6 took 1,791, 1,714 and
// 1,676 us, with the tile in LDS, loaded one tile ahead, 1,684, and the same at 61,441
// targets 964 (4 ahead) and 937.  Without near tiles it would take 1,404.
// Sources per FP32 partial sum.  Sources in spatial order push a partial sum in one
// direction, so it rounds more than one over scattered sources: with 256 per partial
// the 100^2 plane velocity was off by 1.05e-7 against 6.1e-8 in the caller's order.
constexpr int NEAR_FOLD = 64;

template <class N, bool SELF>
__device__ __forceinline__ void near_source(const Vec4<float>& t, int tid, const float* sv, float p[N::NOUT]) {
  W4<float> w;
  N::arg(t, sv, w);
  const float f = N::trans(w);
  const bool mine = SELF && rec_index(sv, N::IDX) == tid;
  if (SELF && __any(mine)) {
    float tmp[N::NOUT];
#pragma unroll
    for (int k = 0; k < N::NOUT; ++k) tmp[k] = 0.f;
    N::acc(sv, w, f, tmp);
#pragma unroll
    for (int k = 0; k < N::NOUT; ++k) p[k] += mine ? 0.f : tmp[k];
  } else {
    N::acc(sv, w, f, p);
  }
}

// `rec`: the tile's records in LDS, two 16-byte words each.
template <class N, bool SELF>
__device__ __forceinline__ void near_tile(const Vec4<float>& t, int tid, const float4* rec, int count,
                                          double S[N::NOUT]) {
  constexpr int NO = N::NOUT;
  for (int j0 = 0; j0 < count; j0 += NEAR_FOLD) {
    const int j1 = min(count, j0 + NEAR_FOLD);
    float p[NO];
#pragma unroll
    for (int k = 0; k < NO; ++k) p[k] = 0.f;
#pragma unroll 4
    for (int j = j0; j < j1; ++j) {
      const float4 lo = rec[2 * j], hi = rec[2 * j + 1];
      const float sv[SREC] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      near_source<N, SELF>(t, tid, sv, p);
    }
#pragma unroll
    for (int k = 0; k < NO; ++k) S[k] += (double)p[k];
  }
}

// One step: 16 staged sources against the wave's column tiles.
template <class P>
struct FarStep {
  u32x4 a;
  f32x4 w, w2;
  __device__ __forceinline__ void read(const typename FarStageOf<P>::T& st, int s, int lane, int wl, int grp) {
    a = st.frag[s * 64 + lane];
    w = st.wgt[s * 16 + wl];
    if constexpr (kSwe<P>) w2 = st.wgt2[s * 16 + wl];
    if constexpr (P::NW == 2) w2 = st.wgt[s * 16 + grp * 4 + 1];
  }
  // D: FAR_COLS accumulators; the shallow-water sums have 3 FAR_COLS (f with the
  // first weights, f^2 with both)
  __device__ __forceinline__ void add(const u32x4 B[FAR_COLS], f32x4* D) const {
    f32x4 r[FAR_COLS];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < FAR_COLS; ++c)
      r[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, B[c]),
                                                     f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
    for (int c = 0; c < FAR_COLS; ++c)
#pragma unroll
      for (int v = 0; v < 4; ++v) r[c][v] = P::trans(r[c][v]);
    if constexpr (P::NW == 0) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int c = 0; c < FAR_COLS; ++c) D[c] = __builtin_amdgcn_mfma_f32_4x4x1f32(w[v], r[c][v], D[c], 0, 0, 0);
      if constexpr (kSwe<P>) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < FAR_COLS; ++c) r[c] *= r[c];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int c = 0; c < FAR_COLS; ++c) {
            f32x4 &D1 = D[FAR_COLS + c], &D2 = D[2 * FAR_COLS + c];
            D1 = __builtin_amdgcn_mfma_f32_4x4x1f32(w[v], r[c][v], D1, 0, 0, 0);
            D2 = __builtin_amdgcn_mfma_f32_4x4x1f32(w2[v], r[c][v], D2, 0, 0, 0);
          }
      }
    } else {
#pragma unroll
      for (int c = 0; c < FAR_COLS; ++c)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          D[c][0] = fmaf(r[c][v], w[v], D[c][0]);
          if constexpr (P::NW == 2) D[c][1] = fmaf(r[c][v], w2[v], D[c][1]);
        }
    }
  }
};

// One block's work: targets [t_block, t_block + 256) of the record array tg[0, nt)
// (particle index order[local]), 64 to a wave, against the ns sources of src in
// groups of FAR_FOLD: group first_group and every group_step-th after it, so that
// the near tiles, which lie together in spatial order, spread over the splits.
// smeta[k] is the ball of sources [k, k + 1) FAR_TILE.  FP64 results go to
// out[k * out_stride + i].
template <class P>
__device__ __forceinline__ void far_block(const Vec4<float>* __restrict__ tg, int nt, int t_block,
                                          const int* __restrict__ order, const float4 tm, const float* __restrict__ src,
                                          const float4* __restrict__ smeta, int ns, int first_group,
                                          int group_step, double* __restrict__ out, int out_stride,
                                          typename FarStageOf<P>::T* stage, float reach = 0.f) {
  using N = typename P::Near;
  constexpr int NO = N::NOUT;
  constexpr int NACC = P::NW == 0 ? 4 : P::NW;
  constexpr int ND = kSwe<P> ? 3 * FAR_COLS : FAR_COLS;  // accumulators
  constexpr int NFAR = kSwe<P> ? 12 : NACC;              // far sums of a target
  auto is_far = [&](const float4& sm) {
    if constexpr (kSwe<P>)
      return tiles_far_swe(tm, sm, reach);
    else
      return tiles_far(tm, sm);
  };
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int grp = lane >> 4;
  const int t_begin = t_block + wid * 64;
  const int i = t_begin + lane;
  const Vec4<float> t = tg[i < nt ? i : nt - 1];
  const int tid = order[i < nt ? i : nt - 1];
  double near_sum[NO];
#pragma unroll
  for (int k = 0; k < NO; ++k) near_sum[k] = 0.0;

  // this split's tiles, in order
  auto next_tile = [&](int jt) {
    jt += FAR_TILE;
    return jt % FAR_FOLD ? jt : jt + (group_step - 1) * FAR_FOLD;
  };
  const int j_begin = first_group * FAR_FOLD;

  float rec[SREC];
  bool have;
  auto load = [&](int jt) {  // this thread's source of the tile at jt
    const int j = jt + (int)threadIdx.x;
    have = j < ns;
    const float4* r = reinterpret_cast<const float4*>(src + (size_t)(have ? j : ns - 1) * SREC);
    const float4 lo = r[0], hi = r[1];
    rec[0] = lo.x, rec[1] = lo.y, rec[2] = lo.z, rec[3] = lo.w;
    rec[4] = hi.x, rec[5] = hi.y, rec[6] = hi.z, rec[7] = hi.w;
  };
  int buf = 0;
  int n_far = 0;
  // near tiles first, through the stages' memory.  Here and below one barrier a tile: a
  // wave writes a buffer again only after the barrier of the tile between, which every
  // wave reaches after its reads of this one.
  if constexpr (kSwe<P>) {
    for (int jt = j_begin; jt < ns; jt = next_tile(jt)) n_far += is_far(smeta[jt / FAR_TILE]) ? 1 : 0;
  } else {
    auto next_near = [&](int jt) {
      while (jt < ns && is_far(smeta[jt / FAR_TILE])) {
        jt = next_tile(jt);
        ++n_far;
      }
      return jt;
    };
    int jt = next_near(j_begin);
    if (jt < ns) load(jt);
    while (jt < ns) {  // block-uniform
      float4* st = reinterpret_cast<float4*>(&stage[buf]);
      st[2 * threadIdx.x] = make_float4(rec[0], rec[1], rec[2], rec[3]);
      st[2 * threadIdx.x + 1] = make_float4(rec[4], rec[5], rec[6], rec[7]);
      const int jn = next_near(next_tile(jt));
      if (jn < ns) load(jn);
      __syncthreads();
      if (t_begin < nt) {
        const float4 sm = smeta[jt / FAR_TILE];
        const int count = min(FAR_TILE, ns - jt);
        if (balls_touch(ball_d2(tm, sm), tm, sm))
          near_tile<N, true>(t, tid, st, count, near_sum);
        else
          near_tile<N, false>(t, tid, st, count, near_sum);
      }
      buf ^= 1;
      jt = jn;
    }
  }

  double far_sum[NFAR];
#pragma unroll
  for (int k = 0; k < NFAR; ++k) far_sum[k] = 0.0;
  double sum[FAR_COLS][NACC];
#pragma unroll
  for (int c = 0; c < FAR_COLS; ++c)
#pragma unroll
    for (int k = 0; k < NACC; ++k) sum[c][k] = 0.0;
  const float X[3] = {t.a - tm.x, t.b - tm.y, P::DIMS == 3 ? t.c - tm.z : 0.f};
  // A weight w times a position, or its square, leaves the normal numbers long before
  // the all-pairs kernel's w / d^2 does (at lengths of 1e-13, of 1e18, or of 1e-6 with weak
  // fields).  In units of the first far tile's distance, a power of two, w / d comes
  // before the product, which lies between w and w / d^2; results keep their bits.
  float unit = 1.f;

  if (n_far > 0) {  // block-uniform
    const float n2t = fmaf(X[0], X[0], fmaf(X[1], X[1], fmaf(X[2], X[2], P::E ? t.d : 0.f)));
    u32x4 B[FAR_COLS];
#pragma unroll
    for (int c = 0; c < FAR_COLS; ++c) {
      // lane (group g, column l % 16) holds coordinate g (or the norm) of target 16 c + l % 16
      const int from = 16 * c + (lane & 15);
      const float a0 = __shfl(X[0], from), a1 = __shfl(X[1], from), a2 = __shfl(X[2], from), a3 = __shfl(n2t, from);
      const float v = grp == 0 ? a0 : grp == 1 ? a1 : grp == 2 ? a2 : a3;
      B[c] = frag_tgt(v, grp == 3);
    }
    f32x4 D[ND];
#pragma unroll
    for (int c = 0; c < ND; ++c) D[c] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto next_far = [&](int jt) {
      while (jt < ns && !is_far(smeta[jt / FAR_TILE])) jt = next_tile(jt);
      return jt;
    };
    int jt = next_far(j_begin);
    load(jt);
    unit = inverse_length(ball_d2(tm, smeta[jt / FAR_TILE]));
    while (jt < ns) {
      typename FarStageOf<P>::T& st = stage[buf];
      {
        // this thread's source: row threadIdx % 16 of step threadIdx / 16; past the
        // end a source of weight 0 at distance 1
        float d[3] = {rec[0] - tm.x, rec[1] - tm.y, P::DIMS == 3 ? rec[2] - tm.z : 0.f};
        float n2 = fmaf(d[0], d[0], fmaf(d[1], d[1], fmaf(d[2], d[2], P::E ? rec[3] : 0.f)));
        float w0 = rec[P::W0], w1 = rec[P::W1];
        if (!have) d[0] = d[1] = d[2] = w0 = w1 = 0.f, n2 = 1.f;
        const int s = threadIdx.x >> 4, r = threadIdx.x & 15;
        st.frag[s * 64 + r] = frag_src(-2.f * d[0]);
        st.frag[s * 64 + 16 + r] = frag_src(-2.f * d[1]);
        st.frag[s * 64 + 32 + r] = frag_src(-2.f * d[2]);
        st.frag[s * 64 + 48 + r] = frag_src_norm(n2);
        float* w = reinterpret_cast<float*>(st.wgt + s * 16 + (r >> 2) * 4) + (r & 3);
        if constexpr (kSwe<P>) {
          // c, c conj(Z); c conj(Z)^2
          float* wb = reinterpret_cast<float*>(st.wgt2 + s * 16 + (r >> 2) * 4) + (r & 3);
          const float a0 = w0 * unit, a1 = w1 * unit;
          const float vr = fmaf(a0, d[0], a1 * d[1]), vi = fmaf(a1, d[0], -a0 * d[1]);
          const float br = vr * unit, bi = vi * unit;
          w[0] = w0;
          w[4] = w1;
          w[8] = vr;
          w[12] = vi;
          wb[0] = fmaf(br, d[0], bi * d[1]);
          wb[4] = fmaf(bi, d[0], -br * d[1]);
          wb[8] = wb[12] = 0.f;
        } else if constexpr (P::NW == 0) {
          const float a0 = w0 * unit;
          w[0] = a0 * d[0];
          w[4] = a0 * d[1];
          w[8] = a0 * d[2];
          w[12] = w0;
        } else {
          w[0] = w0;
          if constexpr (P::NW == 2) w[4] = w1;
        }
      }
      const int jn = next_far(next_tile(jt));
      if (jn < ns) load(jn);
      __syncthreads();
      // two register sets in turn: the next step's LDS reads run under this step
      const int wl = grp * 4 + (P::NW == 0 ? lane & 3 : 0);
      FarStep<P> s0, s1;
      s0.read(st, 0, lane, wl, grp);
#pragma unroll 1
      for (int s = 0; s < 16; s += 2) {
        s1.read(st, s + 1, lane, wl, grp);
        s0.add(B, D);
        s0.read(st, s < 14 ? s + 2 : 15, lane, wl, grp);
        s1.add(B, D);
      }
      // fold at fixed places of the source array, so that the split leaves no trace
      // beyond FP64 rounding
      if (jn >= ns || jn / FAR_PART != jt / FAR_PART) {
        if constexpr (kSwe<P>) {
          // FP64 sums of all four columns would take 96 registers: add the four row
          // groups here, each group keeping one column tile
          const bool hi = grp & 2, odd = grp & 1;
#pragma unroll
          for (int k = 0; k < NFAR; ++k) {
            f32x4* d = D + (k >> 2) * FAR_COLS;
            const int e = k & 3;
            const float k0 = hi ? d[2][e] : d[0][e], k1 = hi ? d[3][e] : d[1][e];
            const float s0 = hi ? d[0][e] : d[2][e], s1 = hi ? d[1][e] : d[3][e];
            const double a = (double)k0 + (double)__shfl_xor(s0, 32), b = (double)k1 + (double)__shfl_xor(s1, 32);
            far_sum[k] += (odd ? b : a) + __shfl_xor(odd ? a : b, 16);
#pragma unroll
            for (int c = 0; c < FAR_COLS; ++c) d[c][e] = 0.f;
          }
        } else {
#pragma unroll
          for (int c = 0; c < FAR_COLS; ++c)
#pragma unroll
            for (int k = 0; k < NACC; ++k) {
              sum[c][k] += (double)D[c][k];
              D[c][k] = 0.f;
            }
        }
      }
      buf ^= 1;
      jt = jn;
    }
  }

  // add the four row groups, then give lane l target t_begin + l its column tile
  if (!kSwe<P> && n_far > 0) {
#pragma unroll
    for (int c = 0; c < FAR_COLS; ++c)
#pragma unroll
      for (int k = 0; k < NACC; ++k) {
        double v = sum[c][k];
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        if (grp == c) far_sum[k] = v;
      }
  }
  if (i < nt) {
    double o[NO];
    const double length = 1.0 / unit;
    if constexpr (kSwe<P>) {
      const double* u1 = far_sum;     // f c, f c conj(Z)
      const double* u2 = far_sum + 4;  // f^2 c, f^2 c conj(Z), f^2 c conj(Z)^2
      const double x = (double)X[0] * unit, y = (double)X[1] * unit, xx = x * x - y * y, xy = 2.0 * x * y;
      o[0] = (x * u1[1] - y * u1[0] - u1[3]) * length;
      o[1] = (x * u1[0] + y * u1[1] - u1[2]) * length;
      o[2] = -(xx * u2[1] - xy * u2[0] - 2.0 * (x * u2[3] - y * u2[2]) + u2[5]) * (length * length);
      o[3] = -(xx * u2[0] + xy * u2[1] - 2.0 * (x * u2[2] + y * u2[3]) + u2[4]) * (length * length);
      o[4] = 0.0;
    } else if constexpr (P::NW == 0) {
      double v[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) v[k] = (double)X[k] * far_sum[3] - far_sum[k] * length;
      if constexpr (P::DIMS == 3) {
#pragma unroll
        for (int k = 0; k < 3; ++k) o[k] = v[k];
      } else {  // PlaneBS accumulates (y, x) separations
        o[0] = v[1];
        o[1] = v[0];
      }
    } else {
#pragma unroll
      for (int k = 0; k < NO; ++k) o[k] = far_sum[k];
    }
#pragma unroll
    for (int k = 0; k < NO; ++k) out[(size_t)k * out_stride + i] = near_sum[k] + o[k];
  }
}

template <class P>
static __global__ __launch_bounds__(256, P::BLOCKS) void far_sum_kernel(const void* __restrict__ tgt, const void* __restrict__ srcv,
                                                         double* __restrict__ partial,
                                                         const float4* __restrict__ tmeta,
                                                         const float4* __restrict__ smeta,
                                                         const int* __restrict__ order, PairArgs a) {
  __shared__ typename FarStageOf<P>::T stage[2];
  const int nblk_t = (a.nt + FAR_TILE - 1) / FAR_TILE;
  const int split = blockIdx.x / nblk_t;
  const int tb = blockIdx.x - split * nblk_t;
  far_block<P>(reinterpret_cast<const Vec4<float>*>(tgt), a.nt, tb * FAR_TILE, order, tmeta[tb],
               reinterpret_cast<const float*>(srcv), smeta, a.ns, split, a.nsplit,
               partial + (size_t)split * P::Near::NOUT * a.nt, a.nt, stage, a.reach);
}

// Batched problems: a persistent launch whose blocks take (problem, target block,
// split) items from a counter until the list is exhausted.
template <class P>
static __global__ __launch_bounds__(256, 4) void far_batch_kernel(
    const void* __restrict__ tgt, const void* __restrict__ srcv, double* __restrict__ partial,
    const float4* __restrict__ tballs, const float4* __restrict__ sballs, const int* __restrict__ order,
    const BatchProblem* __restrict__ probs, const BatchItem* __restrict__ items, int n_items,
    unsigned int* __restrict__ counter) {
  __shared__ FarStage stage[2];
  // the item number passes through a stage: one more word of LDS would leave room
  // for 3 blocks per CU instead of 4
  volatile int* next = reinterpret_cast<volatile int*>(stage);
  for (;;) {
    __syncthreads();  // every wave is done with the last item's stages
    if (threadIdx.x == 0) *next = (int)atomicAdd(counter, 1u);
    __syncthreads();
    const int item = __builtin_amdgcn_readfirstlane(*next);
    __syncthreads();
    if (item >= n_items) break;
    const BatchItem it = items[item];
    const BatchProblem pr = probs[it.prob];
    far_block<P>(reinterpret_cast<const Vec4<float>*>(tgt) + pr.t_off, pr.nt, it.wtile * FAR_TILE, order + pr.t_off,
                 tballs[pr.tball_off + it.wtile], reinterpret_cast<const float*>(srcv) + (size_t)pr.s_off * SREC,
                 sballs + pr.sball_off, pr.ns, it.split, pr.nsplit,
                 partial + pr.part_off + (size_t)it.split * P::Near::NOUT * pr.nt, pr.nt, stage);
  }
}

}  // namespace lpm
