// mlp_kernels.hpp -- the far-field surrogate network on gfx950.
//
// Network: nin -> width (act) -> ... (nhidden act layers) -> nout, act = tanh or
// ISRU x / sqrt(1 + x^2), parameters per layer W[out][in] (row-major) then
// b[out], FP32 master copy.
//
// Training path (FP32 matrix instructions): tiled GEMMs C = A op(B) with the
// bias + activation, the activation's derivative or the bias gradient fused in, and Adam.
// Inference path (FP16 MFMA, FP32 accumulate), specialised for the
// 13 -> 128 -> 128 -> 128 -> 3 surrogate: activations are kept transposed
// (features = MFMA rows, samples = MFMA columns), so the D registers of one
// layer (lane l: rows 4(l/16)+v of each 16-row tile, column l%16) are, after
// bias + activation + FP16 conversion, exactly the B operand of the next layer once
// the next layer's weight fragments are stored with the matching K order:
// k-slot e of lane group g in k-step ks is feature 32 ks + 16 (e/4) + 4 g + e%4.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lpm {

// Inference operands are FP16: the same MFMA rate as BF16 on gfx950 (measured:
// equal launch times) with 3 more mantissa bits, which cut the forward pass's
// error against FP64 from 4.5e-3 to 6e-4 (relative RMS).
typedef _Float16 mlp_t;
typedef mlp_t mlpx8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ floatx4_t mfma16(mlpx8_t a, mlpx8_t b, floatx4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float tanh_fast(float x) {
  // tanh x = 1 - 2 / (exp(2x) + 1), exp via v_exp_f32 (2^y); saturates cleanly
  const float e = __builtin_amdgcn_exp2f(2.8853900817779268f * x);  // 2 log2(e) x
  return 1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f);
}

// Hidden-layer activations: 1 tanh, 2 ISRU x / sqrt(1 + x^2) (one transcendental,
// v_rsq_f32, instead of tanh's two).
constexpr int kActTanh = 1;
constexpr int kActIsru = 2;

template <int ACT>
__device__ __forceinline__ float act_fast(float x) {
  if constexpr (ACT == kActIsru)
    return x * __builtin_amdgcn_rsqf(fmaf(x, x, 1.0f));
  else
    return tanh_fast(x);
}

// Scale of the hidden layers' pre-activations in the MFMA path: with ISRU the
// hidden weights and biases are stored times kIsruScale, so the accumulators
// hold y = x kIsruScale and ISRU(x) = y / sqrt(y^2 + kIsruScale^2), evaluated
// in packed FP16 (v_pk_fma_f16, v_rsq_f16, v_pk_mul_f16) without overflow of
// y^2 for |x| < 16,000.
constexpr float kIsruScale = 1.0f / 64.0f;

// Activation of 8 accumulator values (lo: one 16-row tile's 4, hi: the next
// tile's 4) into the next layer's 8-element B operand.
template <int ACT>
__device__ __forceinline__ mlpx8_t act8(floatx4_t lo, floatx4_t hi) {
  mlpx8_t v;
  if constexpr (ACT == kActIsru) {
    const _Float16 c = (_Float16)(kIsruScale * kIsruScale);
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const float a = p < 2 ? lo[2 * p] : hi[2 * p - 4], b = p < 2 ? lo[2 * p + 1] : hi[2 * p - 3];
      const half2_t y = {(_Float16)a, (_Float16)b};
      const half2_t t = y * y + (half2_t){c, c};
      half2_t r;
      r[0] = __builtin_amdgcn_rsqh(t[0]);
      r[1] = __builtin_amdgcn_rsqh(t[1]);
      const half2_t h = y * r;
      v[2 * p] = h[0];
      v[2 * p + 1] = h[1];
    }
    return v;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (mlp_t)act_fast<ACT>(e < 4 ? lo[e] : hi[e - 4]);
  return v;
}

// Scale the MFMA path applies to the hidden layers' weights and biases.
__host__ __device__ inline float mlp_hidden_scale(int act) {
  return act == kActIsru ? kIsruScale : 1.0f;
}

// ------------------------------------------------------------ FP32 GEMM
// C[M][N] = act(sum_k A(m, k) B(k, n) + bias[n]), with A(m, k) = TA ? A[k][m] :
// A[m][k] and B(k, n) = TB ? B[n][k] : B[k][n]; with H, the product is instead
// multiplied by the activation's derivative at the output H[m][n] (leading
// dimension ldc).  sums (TA only) receives sum_k A(m, k), the bias gradient.
//
// 64 x 64 tile per 256-thread block on the FP32 matrix instruction
// v_mfma_f32_16x16x4_f32: each of the 4 waves holds 32 x 32 outputs as four
// accumulators.  Operands are staged as [row][k] in two LDS buffers of 32 k
// each, the next tile's global loads in flight during the current tile's
// products.  Lane group g = lane / 16 reads k = 4 g .. 4 g + 3 of a 16-k block in one
// ds_read_b128 and step s multiplies its element s, for A and B alike, so a
// block needs 4 LDS reads per 16 matrix instructions; a row pitch of 36
// floats spreads the reads over the banks.  B's rows are the instruction's
// rows: a lane's four results are four consecutive n, one 16-byte store.
// Split K: with part != nullptr, block z covers k in [z kchunk, (z+1) kchunk)
// and writes its partial product (and, after it, its partial sums) to
// part[z][M N (+ M)]; gemm_splitk_reduce adds them in a fixed order.
// At 32,768 samples and width 128 (1.07 GFLOP, 6.8 us of matrix time; the
// operands' 34 MB take 7 us) a layer's forward takes 22 us, its input gradient
// 19.5 and its weight and bias gradient 24 with the reduction; the same on the
// vector units, with the derivative and the sums in kernels of their own, took
// 51, 52 and 188.  What is left is the serial load, product, store of a block
// with 4 K tiles.
constexpr int kGemmTile = 64;
constexpr int kGemmK = 32;
constexpr int kGemmPitch = kGemmK + 4;

struct GemmArgs {
  const float* A;
  const float* B;
  float* C;
  const float* bias;
  const float* H;
  float* sums;
  int M, N, K;
  int lda, ldb, ldc;
  int act;  // 0 none, kActTanh, kActIsru
  float* part;
  int kchunk;
};

// dZ = dH act'(Z) from the output H alone: tanh' = 1 - H^2;
// ISRU' = (1 + Z^2)^(-3/2) = (1 - H^2)^(3/2)
__device__ __forceinline__ float act_slope(int act, float h) {
  const float t = 1.0f - h * h;
  return act == kActIsru ? t * sqrtf(fmaxf(t, 0.0f)) : t;
}

// Eight floats of one operand's 64 x 32 tile (rows r0 .., k0 ..) for this thread.
// ROWS (k contiguous in memory): rows t/8 and t/8 + 32, k = 4 (t%8) .. + 3.
// Else (rows contiguous): row t%64, k = 4 (t/64) .. + 3 and the same + 16.
// Rows past the end repeat the last one (their outputs are not stored), k past
// the end is zero; every load is unconditional, so all are in flight together.
// vec: the k-contiguous rows start on 16 bytes.
template <bool ROWS>
__device__ __forceinline__ void gemm_fetch(const float* __restrict__ X, int ld, int rows, int ke, int r0, int k0,
                                           bool vec, floatx4_t v[2]) {
  const int t = threadIdx.x;
  const bool full = k0 + kGemmK <= ke;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = min(ROWS ? r0 + (t >> 3) + 32 * j : r0 + (t & 63), rows - 1);
    const int k = ROWS ? k0 + 4 * (t & 7) : k0 + 4 * (t >> 6) + 16 * j;
    const float* x = ROWS ? X + (size_t)r * ld : X + r;
    const size_t step = ROWS ? 1 : (size_t)ld;
    if (full) {
      if (ROWS && vec) {
        v[j] = *reinterpret_cast<const floatx4_t*>(x + k);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][e] = x[(size_t)(k + e) * step];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float y = x[(size_t)min(k + e, ke - 1) * step];
        v[j][e] = k + e < ke ? y : 0.f;
      }
    }
  }
}

template <bool ROWS>
__device__ __forceinline__ void gemm_stage(float* __restrict__ S, const floatx4_t v[2]) {
  const int t = threadIdx.x;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = ROWS ? (t >> 3) + 32 * j : (t & 63);
    const int k = ROWS ? 4 * (t & 7) : 4 * (t >> 6) + 16 * j;
    *reinterpret_cast<floatx4_t*>(S + r * kGemmPitch + k) = v[j];
  }
}

template <bool TA, bool TB>
__global__ __launch_bounds__(256) void gemm_f32(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) float As[2][kGemmTile * kGemmPitch];
  __shared__ __attribute__((aligned(16))) float Bs[2][kGemmTile * kGemmPitch];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i16 = lane & 15, g4 = lane >> 4;
  const int m0 = blockIdx.x * kGemmTile, n0 = blockIdx.y * kGemmTile;
  const int wm = 32 * (w & 1), wn = 32 * (w >> 1);
  const int kb = g.part ? (int)blockIdx.z * g.kchunk : 0;
  const int ke = g.part ? min(g.K, kb + g.kchunk) : g.K;
  const bool va = !TA && (g.lda & 3) == 0 && (reinterpret_cast<uintptr_t>(g.A) & 15) == 0;
  const bool vb = TB && (g.ldb & 3) == 0 && (reinterpret_cast<uintptr_t>(g.B) & 15) == 0;
  const bool sums = TA && g.sums && n0 == 0;
  floatx4_t acc[2][2] = {};  // [n tile][m tile]
  floatx4_t fa[2], fb[2];
  float sum = 0.f;
  gemm_fetch<!TA>(g.A, g.lda, g.M, ke, m0, kb, va, fa);
  gemm_fetch<TB>(g.B, g.ldb, g.N, ke, n0, kb, vb, fb);
  int cur = 0;
  for (int k0 = kb; k0 < ke; k0 += kGemmK, cur ^= 1) {
    gemm_stage<!TA>(As[cur], fa);
    gemm_stage<TB>(Bs[cur], fb);
    if (sums) {
      const floatx4_t s = fa[0] + fa[1];
      sum += (s[0] + s[1]) + (s[2] + s[3]);
    }
    __syncthreads();  // also: every wave has left the buffer staged next
    if (k0 + kGemmK < ke) {
      gemm_fetch<!TA>(g.A, g.lda, g.M, ke, m0, k0 + kGemmK, va, fa);
      gemm_fetch<TB>(g.B, g.ldb, g.N, ke, n0, k0 + kGemmK, vb, fb);
    }
    const float* a = As[cur] + (wm + i16) * kGemmPitch + 4 * g4;
    const float* b = Bs[cur] + (wn + i16) * kGemmPitch + 4 * g4;
#pragma unroll
    for (int kk = 0; kk < kGemmK; kk += 16) {
      floatx4_t av[2], bv[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        av[q] = *reinterpret_cast<const floatx4_t*>(a + 16 * q * kGemmPitch + kk);
        bv[q] = *reinterpret_cast<const floatx4_t*>(b + 16 * q * kGemmPitch + kk);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int q = 0; q < 2; ++q)
            acc[p][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[p][s], av[q][s], acc[p][q], 0, 0, 0);
    }
  }
  const size_t mn = (size_t)g.M * g.N;
  float* P = g.part ? g.part + (size_t)blockIdx.z * (mn + (g.sums ? g.M : 0)) : nullptr;
  if (sums) {  // 4 waves' sums of each row, in order; the staging buffers are free after the barrier
    __syncthreads();
    As[0][threadIdx.x] = sum;
    __syncthreads();
    const int m = m0 + threadIdx.x;
    if (threadIdx.x < kGemmTile && m < g.M) {
      const float s = (As[0][threadIdx.x] + As[0][threadIdx.x + 64]) +
                      (As[0][threadIdx.x + 128] + As[0][threadIdx.x + 192]);
      (P ? P + mn : g.sums)[m] = s;
    }
  }
  float* C = P ? P : g.C;
  const int ldc = P ? g.N : g.ldc;
  const bool vc = (ldc & 3) == 0 && ((reinterpret_cast<uintptr_t>(C) | reinterpret_cast<uintptr_t>(g.H)) & 15) == 0;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int m = m0 + wm + 16 * q + i16, n = n0 + wn + 16 * p + 4 * g4;
      if (m >= g.M || n >= g.N) continue;
      const size_t at = (size_t)m * ldc + n;
      const int cols = min(4, g.N - n);
      floatx4_t v = acc[p][q];
      if (!P) {
        if (g.bias)
          for (int e = 0; e < cols; ++e) v[e] += g.bias[n + e];
        if (g.H) {
          floatx4_t h = {};
          if (vc && cols == 4) h = *reinterpret_cast<const floatx4_t*>(g.H + at);
          else
            for (int e = 0; e < cols; ++e) h[e] = g.H[at + e];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] *= act_slope(g.act, h[e]);
        } else if (g.act == kActTanh) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = tanhf(v[e]);
        } else if (g.act == kActIsru) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = v[e] / sqrtf(fmaf(v[e], v[e], 1.0f));
        }
      }
      if (vc && cols == 4) *reinterpret_cast<floatx4_t*>(C + at) = v;
      else
        for (int e = 0; e < cols; ++e) C[at + e] = v[e];
    }
  }
}

// out[t] = sum over splits z of part[z][t]: 64 outputs per block, wave w adds
// splits w, w + 4, ... with 8 loads in flight, then the four waves' sums (fixed order).
static __global__ __launch_bounds__(256) void gemm_splitk_reduce(int splits, int n, const float* __restrict__ part,
                                                                float* __restrict__ out) {
  __shared__ float sh[256];
  const int w = threadIdx.x >> 6, t = blockIdx.x * 64 + (threadIdx.x & 63);
  float s = 0.f;
  if (t < n) {
    int z = w;
    for (; z + 28 < splits; z += 32) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = part[(size_t)(z + 4 * e) * n + t];
#pragma unroll
      for (int e = 0; e < 8; ++e) s += v[e];
    }
    for (; z < splits; z += 4) s += part[(size_t)z * n + t];
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  if (w == 0 && t < n) out[t] = (sh[threadIdx.x] + sh[threadIdx.x + 64]) + (sh[threadIdx.x + 128] + sh[threadIdx.x + 192]);
}

// ------------------------------------------------------- FP16 MFMA forward
// Weight fragments, staged once per block in LDS:
//   W1: [8 rt][64 lanes][8]      (K = 32, inputs 0..nin-1, zero padded)
//   W2, W3: [8 rt][4 ks][64][8]  (K order permuted as described above)
//   W4: [4 ks][64][8]            (rows 0..nout-1 of one 16-row tile)
// bias: b1, b2, b3 (128 each), b4 (16), FP32.
constexpr int kW1Frag = 8 * 64 * 8;
constexpr int kWHFrag = 8 * 4 * 64 * 8;
constexpr int kW4Frag = 4 * 64 * 8;
constexpr int kMlpFragElems = kW1Frag + 2 * kWHFrag + kW4Frag;  // FP16 elements
constexpr int kMlpBiasElems = 128 * 3 + 16;

__host__ __device__ inline int hidden_k_feature(int ks, int g, int e) {
  return 32 * ks + 16 * (e / 4) + 4 * g + (e % 4);
}

// Convert FP32 parameters (13 -> 128 x3 -> 3 layout) into fragment order.
static __global__ __launch_bounds__(256) void mlp_pack_fragments(const float* __restrict__ P, int nin, int nout,
                                                         mlp_t* __restrict__ frag,
                                                         float* __restrict__ bias, float hscale) {
  const int W = 128;
  const float* W1 = P;
  const float* b1 = W1 + W * nin;
  const float* W2 = b1 + W;
  const float* b2 = W2 + W * W;
  const float* W3 = b2 + W;
  const float* b3 = W3 + W * W;
  const float* W4 = b3 + W;
  const float* b4 = W4 + nout * W;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < kMlpFragElems; t += gridDim.x * blockDim.x) {
    float v = 0.f;
    if (t < kW1Frag) {
      const int rt = t / 512, l = (t / 8) % 64, e = t % 8;
      const int row = 16 * rt + l % 16, k = 8 * (l / 16) + e;
      v = k < nin ? W1[row * nin + k] : 0.f;
    } else if (t < kW1Frag + 2 * kWHFrag) {
      const int u = (t - kW1Frag) % kWHFrag;
      const float* Wm = (t - kW1Frag) < kWHFrag ? W2 : W3;
      const int rt = u / 2048, ks = (u / 512) % 4, l = (u / 8) % 64, e = u % 8;
      v = Wm[(16 * rt + l % 16) * W + hidden_k_feature(ks, l / 16, e)];
    } else {
      const int u = t - kW1Frag - 2 * kWHFrag;
      const int ks = u / 512, l = (u / 8) % 64, e = u % 8;
      const int row = l % 16;
      v = row < nout ? W4[row * W + hidden_k_feature(ks, l / 16, e)] : 0.f;
    }
    frag[t] = (mlp_t)(t < kW1Frag + 2 * kWHFrag ? v * hscale : v);
  }
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < kMlpBiasElems; t += gridDim.x * blockDim.x) {
    float v;
    if (t < 128) v = b1[t] * hscale;
    else if (t < 256) v = b2[t - 128] * hscale;
    else if (t < 384) v = b3[t - 256] * hscale;
    else v = (t - 384) < nout ? b4[t - 384] : 0.f;
    bias[t] = v;
  }
}

// One wavefront evaluates NCT x 16 samples.  in8[ct] holds this lane's 8 input
// features (features 8 g .. 8 g + 7 of sample 16 ct + l % 16, g = l / 16);
// on return out[ct][0..2] are the outputs of that sample in lanes 0..15
// (lanes 16..63 hold padding rows).  Weights/biases in LDS (fragment order);
// sbias must be 16-byte aligned (it is read as float4 rows).
template <int NCT, int ACT = kActTanh>
__device__ __forceinline__ void mlp_wave_forward(const mlpx8_t in8[NCT], const mlp_t* __restrict__ sfrag,
                                                 const float* __restrict__ sbias, float out[NCT][4]) {
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4;
  const mlpx8_t* F1 = reinterpret_cast<const mlpx8_t*>(sfrag);
  const mlpx8_t* F2 = reinterpret_cast<const mlpx8_t*>(sfrag + kW1Frag);
  const mlpx8_t* F3 = reinterpret_cast<const mlpx8_t*>(sfrag + kW1Frag + kWHFrag);
  const mlpx8_t* F4 = reinterpret_cast<const mlpx8_t*>(sfrag + kW1Frag + 2 * kWHFrag);
  floatx4_t acc[8][NCT];
  mlpx8_t h[4][NCT];  // B operands of the next layer: [ks][ct]

  // The accumulators start at the bias (lane group g holds rows 4 g .. 4 g + 3
  // of each 16-row tile), so the MFMA adds it and the activation pass needs no
  // separate add: a fifth of the vector instructions of a forward pass.
  auto bias4 = [&](const float* b, int rt) -> floatx4_t {
    return *reinterpret_cast<const floatx4_t*>(b + 16 * rt + 4 * g);
  };
  // layer 1: K = 32 (one step)
#pragma unroll
  for (int rt = 0; rt < 8; ++rt) {
    const mlpx8_t a = F1[rt * 64 + lane];
    const floatx4_t z = bias4(sbias, rt);
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) acc[rt][ct] = mfma16(a, in8[ct], z);
  }
  // activation -> next B operands
  auto activate = [&]() {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) h[ks][ct] = act8<ACT>(acc[2 * ks][ct], acc[2 * ks + 1][ct]);
  };
  activate();
  // layers 2, 3: 128 x 128
#pragma unroll 1
  for (int layer = 0; layer < 2; ++layer) {
    const mlpx8_t* F = layer == 0 ? F2 : F3;
    const float* bl = sbias + 128 * (layer + 1);
#pragma unroll
    for (int rt = 0; rt < 8; ++rt) {
      const floatx4_t z = bias4(bl, rt);
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) acc[rt][ct] = z;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const mlpx8_t a = F[(rt * 4 + ks) * 64 + lane];
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) acc[rt][ct] = mfma16(a, h[ks][ct], acc[rt][ct]);
      }
    }
    activate();
  }
  // output layer: one 16-row tile, K = 128
  floatx4_t o[NCT];
  const floatx4_t bo = bias4(sbias + 384, 0);
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) o[ct] = bo;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const mlpx8_t a = F4[ks * 64 + lane];
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) o[ct] = mfma16(a, h[ks][ct], o[ct]);
  }
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
    for (int v = 0; v < 4; ++v) out[ct][v] = o[ct][v];
}

}  // namespace lpm
