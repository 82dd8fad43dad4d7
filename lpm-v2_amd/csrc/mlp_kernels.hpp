// mlp_kernels.hpp -- the far-field surrogate network on gfx950.
//
// Network: nin -> width (act) -> ... (nhidden act layers) -> nout, act = tanh or
// ISRU x / sqrt(1 + x^2), parameters per layer W[out][in] (row-major) then
// b[out], FP32 master copy.
//
// Training path (FP32 matrix instructions): all layers forward and all back in one
// launch each, or a tiled GEMM C = A op(B) a layer where they are too wide, the weight
// and bias gradients in one launch, and Adam.
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
// Split K: with part != nullptr, split z covers k in [z kchunk, (z+1) kchunk)
// and writes its partial product (and, after it, its partial sums) to
// part + z part_stride; gemm_splitk_reduce adds them in a fixed order.
// The weight and bias gradients of all layers are one launch (gemm_dw): at 32,768
// samples, 13 -> 128 x 3 -> 3, 768 blocks and 49 us with the reduction (20 us of matrix
// time), against 24 us a layer in launches of their own and 188 on the vector units
// with the sums in a kernel of its own.  Layers up to 128 wide go through mlp_chain
// instead of one product each.
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
  size_t part_stride;
  int kchunk;
};

// dZ = dH act'(Z) from the output H alone: tanh' = 1 - H^2;
// ISRU' = (1 + Z^2)^(-3/2) = (1 - H^2)^(3/2)
__device__ __forceinline__ float act_slope(int act, float h) {
  const float t = 1.0f - h * h;
  return act == kActIsru ? t * sqrtf(fmaxf(t, 0.0f)) : t;
}

// x / sqrt(1 + x^2): the hardware's reciprocal square root with one Newton step, a
// fifth of the 38 instructions of the library's square root and division and as close
// to the exact value.
__device__ __forceinline__ float isru(float x) {
  const float t = fmaf(x, x, 1.0f), r = __builtin_amdgcn_rsqf(t), h = 0.5f * r;
  const float n = fmaf(h, fmaf(-t * r, r, 1.0f), r);
  return x * (t < 1e38f ? n : r);  // t may overflow
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

// One block's 64 x 64 outputs: tile (mb, nb), split z.
struct GemmStage {
  float A[2][kGemmTile * kGemmPitch], B[2][kGemmTile * kGemmPitch];
};

template <bool TA, bool TB>
__device__ __forceinline__ void gemm_block(const GemmArgs& g, int mb, int nb, int z, GemmStage& st) {
  auto& As = st.A;
  auto& Bs = st.B;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i16 = lane & 15, g4 = lane >> 4;
  const int m0 = mb * kGemmTile, n0 = nb * kGemmTile;
  const int wm = 32 * (w & 1), wn = 32 * (w >> 1);
  const int kb = g.part ? z * g.kchunk : 0;
  const int ke = g.part ? min(g.K, kb + g.kchunk) : g.K;
  const bool va = !TA && (g.lda & 3) == 0 && (reinterpret_cast<uintptr_t>(g.A) & 15) == 0;
  const bool vb = TB && (g.ldb & 3) == 0 && (reinterpret_cast<uintptr_t>(g.B) & 15) == 0;
  const bool sums = TA && g.sums && n0 == 0;
  const bool idle = m0 + wm >= g.M || n0 + wn >= g.N;  // a wave of nothing but padding
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
    if (idle) continue;
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
  float* P = g.part ? g.part + z * g.part_stride : nullptr;
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
          for (int e = 0; e < 4; ++e) v[e] = isru(v[e]);
        }
      }
      if (vc && cols == 4) *reinterpret_cast<floatx4_t*>(C + at) = v;
      else
        for (int e = 0; e < cols; ++e) C[at + e] = v[e];
    }
  }
}

template <bool TA, bool TB>
__global__ __launch_bounds__(256) void gemm_f32(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) GemmStage st;
  gemm_block<TA, TB>(g, blockIdx.x, blockIdx.y, blockIdx.z, st);
}

// Weight and bias gradients of all layers, dW_l = dZ_l^T H_(l-1) and db_l = column sums
// of dZ_l: block x is a tile of some layer, block y a split.
constexpr int kMaxLayers = 17;  // 16 hidden layers and the output
struct DwArgs {
  GemmArgs layer[kMaxLayers];
  int first[kMaxLayers + 1];  // first tile of each layer
};

static __global__ __launch_bounds__(256) void gemm_dw(DwArgs a) {
  __shared__ __attribute__((aligned(16))) GemmStage st;
  int l = 0;
  while ((int)blockIdx.x >= a.first[l + 1]) ++l;
  const GemmArgs& g = a.layer[l];
  const int tile = blockIdx.x - a.first[l], mt = (g.M + kGemmTile - 1) / kGemmTile;
  gemm_block<true, false>(g, tile % mt, tile / mt, blockIdx.y, st);
}

// ------------------------------------------------- chains of layers up to 128 wide
// A block takes 16 MT samples through all layers, forward (from the inputs) or
// backward (from the output's gradient to every layer's dZ), its activations in LDS
// between layers and stored once for the products that need them later.  Wave w
// computes columns 32 w .. + 31 with the layer's weights in registers, in the matrix
// instruction's operand order.  As one product a layer, each launch wrote 17 MB that
// the next one read back behind a launch of 4 us: 70 us forward and 56 backward at
// 32,768 samples (16 us of matrix time each), against 47 and 48 here, where a layer's
// loads and stores still alternate with its products (32 samples a block: 58 and 49).
// A training step on 4,096 samples took 133 us and takes 80.
constexpr int kChainWidth = 128;
constexpr int kChainPitch = kChainWidth + 4;

struct ChainArgs {
  int n, nin, width, nout, layers, act;
  const float* P;     // parameters
  const float* X;     // forward: inputs [n][nin]
  const float* dY;    // backward: output gradient [n][nout]
  float* H;           // layer l's output at H + l slot
  float* dZ;          // backward: layer l's dZ at dZ + l slot
  size_t slot;
};

__device__ __forceinline__ int64_t chain_offset(const ChainArgs& a, int l) {
  return l == 0 ? 0 : (int64_t)a.width * a.nin + a.width + (int64_t)(l - 1) * (a.width * (a.width + 1));
}

// 16-k blocks a product of length k is unrolled for.
__host__ __device__ constexpr int chain_blocks(int k) { return k <= 16 ? 1 : k <= 32 ? 2 : k <= 64 ? 4 : 8; }

// LDS rows m0 .. of X [n][k], zero past the end and up to the product's length.
template <int MT>
__device__ __forceinline__ void chain_load(float (*Hs)[kChainPitch], const float* __restrict__ X, int n, int m0, int k) {
  const int blocks = chain_blocks(k), shift = 4 + (blocks > 1) + (blocks > 2) + (blocks > 4);
  for (int t = threadIdx.x; t < (16 * MT) << shift; t += 256) {
    const int r = t >> shift, c = t & ((1 << shift) - 1);
    Hs[r][c] = m0 + r < n && c < k ? X[(size_t)(m0 + r) * k + c] : 0.f;
  }
}

// acc = LDS rows times the wave's 32 columns of B(k, n) = TB ? W[n][k] : W[k][n], for
// K <= 16 KK.  Row r of product p is column n0 + 2 r + p, so that a lane reads W[k][n]
// two columns at a time and its results are eight consecutive columns.  Columns past
// the end repeat the last (they are not kept), k past the end is zero; without a
// branch among them all loads are in flight together.
template <int MT, bool TB, int KK>
__device__ __forceinline__ void chain_product_k(const float (*Hs)[kChainPitch], const float* __restrict__ W, int K,
                                                int N, int n0, floatx4_t acc[MT][2]) {
  const int lane = threadIdx.x & 63, i16 = lane & 15, g4 = lane >> 4;
  typedef float floatx2_t __attribute__((ext_vector_type(2)));
  floatx4_t bv[2][KK];
  const int n = n0 + 2 * i16;
  if (TB && K == 16 * KK && (reinterpret_cast<uintptr_t>(W) & 15) == 0) {
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int p = 0; p < 2; ++p)
        bv[p][kk] = *reinterpret_cast<const floatx4_t*>(W + (size_t)min(n + p, N - 1) * K + 16 * kk + 4 * g4);
  } else if (!TB && (N & 1) == 0 && (reinterpret_cast<uintptr_t>(W) & 7) == 0) {
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = 16 * kk + 4 * g4 + e;
        const floatx2_t y = *reinterpret_cast<const floatx2_t*>(W + (size_t)min(k, K - 1) * N + min(n, N - 2));
        bv[0][kk][e] = k < K ? y[0] : 0.f;
        bv[1][kk][e] = k < K ? y[1] : 0.f;
      }
  } else {
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int k = 16 * kk + 4 * g4 + e, kc = min(k, K - 1), nc = min(n + p, N - 1);
          const float y = TB ? W[(size_t)nc * K + kc] : W[(size_t)kc * N + nc];
          bv[p][kk][e] = k < K ? y : 0.f;
        }
  }
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) {
    floatx4_t av[MT];
#pragma unroll
    for (int q = 0; q < MT; ++q)
      av[q] = *reinterpret_cast<const floatx4_t*>(&Hs[16 * q + i16][16 * kk + 4 * g4]);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int q = 0; q < MT; ++q)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          acc[q][p] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[p][kk][s], av[q][s], acc[q][p], 0, 0, 0);
  }
}

template <int MT, bool TB>
__device__ __forceinline__ void chain_product(const float (*Hs)[kChainPitch], const float* __restrict__ W, int K, int N,
                                              int n0, floatx4_t acc[MT][2]) {
  if (chain_blocks(K) == 1) chain_product_k<MT, TB, 1>(Hs, W, K, N, n0, acc);
  else if (chain_blocks(K) == 2) chain_product_k<MT, TB, 2>(Hs, W, K, N, n0, acc);
  else if (chain_blocks(K) == 4) chain_product_k<MT, TB, 4>(Hs, W, K, N, n0, acc);
  else chain_product_k<MT, TB, 8>(Hs, W, K, N, n0, acc);
}

__device__ __forceinline__ floatx4_t chain_read(const float* __restrict__ row, int n, int N, bool vec) {
  floatx4_t v = {0.f, 0.f, 0.f, 0.f};
  if (vec && n + 4 <= N) v = *reinterpret_cast<const floatx4_t*>(row + n);
  else
    for (int e = 0; e < 4; ++e)
      if (n + e < N) v[e] = row[n + e];
  return v;
}
// The block's rows of a layer's result from LDS to X [n][k].
template <int MT>
__device__ __forceinline__ void chain_store(const float (*Hs)[kChainPitch], float* __restrict__ X, int n, int m0, int k) {
  const int rows = min(16 * MT, n - m0);
  if ((k & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0) {
    const int c = 4 * (threadIdx.x & 31);
    if (c < k)
      for (int r = threadIdx.x >> 5; r < rows; r += 8)
        *reinterpret_cast<floatx4_t*>(X + (size_t)(m0 + r) * k + c) = *reinterpret_cast<const floatx4_t*>(&Hs[r][c]);
  } else {
    for (int r = threadIdx.x >> 5; r < rows; r += 8)
      for (int c = threadIdx.x & 31; c < k; c += 32) X[(size_t)(m0 + r) * k + c] = Hs[r][c];
  }
}

// One layer of mlp_chain: samples m0 .. m0 + 16 MT - 1 (LDS rows Hs), columns n0 ..
// n0 + 31.  idle: the wave has no part in it; zero: but its columns are set to zero.
template <int MT, bool FORWARD>
__device__ __forceinline__ void chain_layer(const ChainArgs& a, float (*Hs)[kChainPitch], int l, int m0, int n0,
                                            bool idle, bool zero) {
  const int lane = threadIdx.x & 63, i16 = lane & 15, g4 = lane >> 4;
  const int last = a.layers - 1;
  const int din = l == 0 ? a.nin : a.width, dout = l == last ? a.nout : a.width;
  const float* W = a.P + chain_offset(a, l);
  const int N = FORWARD ? dout : din;
  const bool vec = (N & 3) == 0 && ((reinterpret_cast<uintptr_t>(a.H) | reinterpret_cast<uintptr_t>(a.dZ)) & 15) == 0 &&
                   (a.slot & 3) == 0;
  floatx4_t acc[MT][2] = {}, h[MT][2], bias[2] = {};
  const int n8 = n0 + 8 * g4;  // the lane's columns n8 .. n8 + 7 of rows 16 q + i16
  if (!idle) {
    if constexpr (FORWARD) {
#pragma unroll
      for (int e = 0; e < 8; ++e) bias[e >> 2][e & 3] = W[(size_t)din * dout + min(n8 + e, N - 1)];
      chain_product<MT, true>(Hs, W, din, N, n0, acc);
    } else {
      // the outputs that the slope needs, under the products
#pragma unroll
      for (int q = 0; q < MT; ++q)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          h[q][c] = chain_read(a.H + (l - 1) * a.slot + (size_t)min(m0 + 16 * q + i16, a.n - 1) * N, n8 + 4 * c, N, vec);
      chain_product<MT, false>(Hs, W, dout, N, n0, acc);
    }
  }
  __syncthreads();  // every wave has read this layer's rows
  if (!idle || zero) {
#pragma unroll
    for (int q = 0; q < MT; ++q)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        floatx4_t v = {acc[q][0][2 * c], acc[q][1][2 * c], acc[q][0][2 * c + 1], acc[q][1][2 * c + 1]};
        if (!idle) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (FORWARD) {
              v[e] += bias[c][e];
              if (l != last) {
                if (a.act == kActTanh) v[e] = tanhf(v[e]);
                else if (a.act == kActIsru) v[e] = isru(v[e]);
              }
            } else {
              v[e] *= act_slope(a.act, h[q][c][e]);
            }
            if (n8 + 4 * c + e >= N) v[e] = 0.f;
          }
        }
        *reinterpret_cast<floatx4_t*>(&Hs[16 * q + i16][n8 + 4 * c]) = v;
      }
  }
  __syncthreads();
}

template <int MT, bool FORWARD>
__global__ __launch_bounds__(256, 2) void mlp_chain(ChainArgs a) {
  __shared__ __attribute__((aligned(16))) float Hs[16 * MT][kChainPitch];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = blockIdx.x * 16 * MT;
  const int last = a.layers - 1;
  chain_load<MT>(Hs, FORWARD ? a.X : a.dY, a.n, m0, FORWARD ? a.nin : a.nout);
  __syncthreads();
  for (int i = 0; i < (FORWARD ? a.layers : last); ++i) {
    const int l = FORWARD ? i : last - i;
    const int N = FORWARD ? (l == last ? a.nout : a.width) : (l == 0 ? a.nin : a.width);
    if (N <= 32)  // a 16-row tile to each wave instead of 32 columns
      chain_layer<1, FORWARD>(a, Hs + 16 * (w % MT), l, m0 + 16 * (w % MT), 0, w >= MT, false);
    else
      chain_layer<MT, FORWARD>(a, Hs, l, m0, 32 * w, 32 * w >= N, true);
    chain_store<MT>(Hs, FORWARD ? a.H + l * a.slot : a.dZ + (l - 1) * a.slot, a.n, m0, N);
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
