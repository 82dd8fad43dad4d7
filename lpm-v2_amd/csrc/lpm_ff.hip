// lpm_ff.hip -- sphere BVE with a learned far field.
//
// Sources are grouped in coarse cells (the particles of a coarse mesh face).
// For each target cell t and source cell s, with cell centroids c, angular
// radii rho and the angle a(t, s) between their centroid directions:
//   near   a < r_near + rho_t + rho_s : direct FP32-compensated sum over s's sources
//   far    otherwise                  : analytic expansion of s to order P (2..4)
//          in its moments M0..MP of w = zeta A about c_s (P = 4: 35 numbers)
//   band   far and a < r_band + rho_t + rho_s : far + the MLP's correction of the
//          expansion's remainder (FP16 MFMA), trained on direct sums
// Cell membership is Lagrangian (fixed at set-up); centroids, radii and
// moments follow the particles and are recomputed at every evaluation.
//
// Velocity assembly, per target x (on the sphere of radius R):
//   u = V x x,  V = sum_near s_ij (x - y_j) + sum_far G_s(x) / (4 pi R)
// with s_ij = -zeta_j A_j / (4 pi R (R^2 - x.y_j)); the parts of V along x drop
// out of V x x.  G_s(x) = sum_j w_j y_j / (R^2 - x.y_j) expanded about c: with
// phi = 1 / D, D = R^2 - x.c (evaluated as (|x-c|^2 + R^2 - |c|^2) / 2) and
// 1 / (D - x.d) = phi sum_k (phi x.d)^k for y = c + d,
//   G_s = c alpha + beta,  alpha = sum_{k=0..P} phi^(k+1) M_k[x,..,x],
//                          beta  = sum_{k=1..P} phi^k M_k[., x,..,x]
// (M_k[., x^(k-1)] the k-th moment tensor contracted k-1 times with x).
//
// Cells are fixed regions: a particle belongs to the cell whose generator (the
// set-up centroid direction of a coarse mesh face) is nearest, and particles
// are binned anew (stable radix sort by cell) at every evaluation, so cells
// keep their size however the flow strains the particles.
//
// The network works in a frame of its cell: e3 along the centroid c, e1 towards
// the cell's anchor direction (fixed at set-up: its source farthest from c),
// e2 = e3 x e1.  Cells of one mesh level then look alike to it, which fixes the
// orientation of the cell's odd moments that the 10 moments leave open.
// Inputs (13): Q (x - c) / l, M0 / W, Q M1 / (W l), Q M2 Q^T / (W l^2) (6), with
// Q the frame rows, l = 2 R sin(rho / 2) and W = sum |w|.  Output o (3, cell
// frame): the expansion's remainder of G_s / (4 pi R) is Q^T o s_out / r^(P+2)
// with r = |x - c| / l and s_out = W / (4 pi R l^2), a scaling under which the
// remainder (~ W l^(P+1) / |x - c|^(P+3)) is O(1) at every distance in the band.
#include <math.h>

#include <algorithm>
#include <numeric>
#include <random>
#include <string>
#include <vector>

#include "lpm_internal.hpp"
#include "lpm_mlp.hpp"
#include "mlp_kernels.hpp"
#include "pair_kernels.hpp"

using lpm::DevBuf;
using lpm::fail;

namespace {

constexpr double kPi = 3.14159265358979323846;
// targets per lane in the near / far kernels.  Wave tiles are per target cell
// (~1,536 targets at L8 with 1,280 cells), so the last tile of a cell is
// partly empty: 96 % of lanes are busy at 2 targets per lane against 92 % at
// 4, and the expansion-mode evaluation at L8 took 23.6 ms against 25.1 ms.
constexpr int kR = 2;
constexpr int kKT = 256;     // sources per compensated tile
constexpr int kNMom = 35;    // moments M0..M4: 1 + 3 + 6 + 10 + 15
constexpr int kCellRec = 40; // floats per far-field cell record
constexpr int kMlpRec = 32;  // floats per MLP cell record
constexpr int kMlpNct = 2;   // 16-target column tiles per network pass
constexpr int kMlpTile = 16 * kMlpNct;  // targets per network work item
// The near and far kernels split their work (near lists, far record lists) in
// up to kSplitMax parts, enough for about kSplitRounds rounds of resident waves.
constexpr double kSplitRounds = 6.0;
constexpr int kSplitMax = 8;

// Symmetric moment tensors are stored by their sorted index tuples in
// lexicographic order: M2 {00 01 02 11 12 22}, M3 {000 001 002 011 012 022 111
// 112 122 222}, M4 {0000 0001 ... 2222}; moment k starts at kMomOff[k].
constexpr int kMomOff[5] = {0, 1, 4, 10, 20};
__host__ __device__ constexpr int sym2(int a, int b) {
  return a <= b ? a * (5 - a) / 2 + b : b * (5 - b) / 2 + a;
}
__host__ __device__ constexpr int sym3(int a, int b, int c) {
  // sort a <= b <= c
  return a > b ? sym3(b, a, c) : (b > c ? sym3(a, c, b) : (a == 0 ? 0 : (a == 1 ? 6 : 9)) + sym2(b, c) - sym2(a, a));
}
__host__ __device__ constexpr int sym4(int a, int b, int c, int d) {
  return a > b ? sym4(b, a, c, d)
               : (b > c ? sym4(a, c, b, d)
                        : (c > d ? sym4(a, b, d, c)
                                 : (a == 0 ? 0 : (a == 1 ? 10 : 14)) + sym3(b, c, d) - sym3(a, a, a)));
}
// unique index tuples of M2, M3, M4 and their multiplicities in a full contraction
constexpr int kPair[6][2] = {{0, 0}, {0, 1}, {0, 2}, {1, 1}, {1, 2}, {2, 2}};
constexpr int kTri[10][3] = {{0, 0, 0}, {0, 0, 1}, {0, 0, 2}, {0, 1, 1}, {0, 1, 2},
                             {0, 2, 2}, {1, 1, 1}, {1, 1, 2}, {1, 2, 2}, {2, 2, 2}};
constexpr int kQuad[15][4] = {{0, 0, 0, 0}, {0, 0, 0, 1}, {0, 0, 0, 2}, {0, 0, 1, 1}, {0, 0, 1, 2},
                              {0, 0, 2, 2}, {0, 1, 1, 1}, {0, 1, 1, 2}, {0, 1, 2, 2}, {0, 2, 2, 2},
                              {1, 1, 1, 1}, {1, 1, 1, 2}, {1, 1, 2, 2}, {1, 2, 2, 2}, {2, 2, 2, 2}};
constexpr float kPairMul[6] = {1, 2, 2, 1, 2, 1};
constexpr float kTriMul[10] = {1, 3, 3, 3, 6, 3, 1, 3, 3, 1};

// Position in m[] of M_k[i, rest] for each free index i and unique tuple `rest`
// of the remaining k-1 indices, tabulated at compile time so that the unrolled
// contractions index the moments with constants.
struct MomIndex {
  int b2[3][3];
  int b3[3][6];
  int b4[3][10];
};
constexpr MomIndex make_mom_index() {
  MomIndex t{};
  for (int k = 0; k < 3; ++k) {
    for (int j = 0; j < 3; ++j) t.b2[k][j] = kMomOff[2] + sym2(k, j);
    for (int p = 0; p < 6; ++p) t.b3[k][p] = kMomOff[3] + sym3(k, kPair[p][0], kPair[p][1]);
    for (int q = 0; q < 10; ++q) t.b4[k][q] = kMomOff[4] + sym4(k, kTri[q][0], kTri[q][1], kTri[q][2]);
  }
  return t;
}
constexpr MomIndex kMomIdx = make_mom_index();

// Expansion of G = sum_j w_j y_j / (R^2 - x.y_j) to order P about c from the
// moments m[35] (T = float: the far kernel, m already divided by 4 pi R;
// T = double: training targets).  D = (|x-c|^2 + e_c) / 2, e_c = R^2 - |c|^2.
__device__ __forceinline__ float recip(float v) { return __builtin_amdgcn_rcpf(v); }
__device__ __forceinline__ double recip(double v) { return 1.0 / v; }

template <int P, typename T>
__device__ __forceinline__ void expansion(const T c[3], T e_c, const T* m, const T x[3], T G[3]) {
  const T dx = x[0] - c[0], dy = x[1] - c[1], dz = x[2] - c[2];
  const T D = T(0.5) * (dx * dx + dy * dy + dz * dz + e_c);
  const T phi = recip(D);
  // b_k = M_k[., x^(k-1)], a_k = x . b_k
  T b[5][3] = {};
  T a[5] = {};
  a[0] = m[0];
#pragma unroll
  for (int k = 0; k < 3; ++k) b[1][k] = m[1 + k];
  if (P >= 2) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      T s = 0;
#pragma unroll
      for (int j = 0; j < 3; ++j) s += m[kMomIdx.b2[k][j]] * x[j];
      b[2][k] = s;
    }
  }
  if (P >= 3) {
    T q[6];
#pragma unroll
    for (int p = 0; p < 6; ++p) q[p] = T(kPairMul[p]) * x[kPair[p][0]] * x[kPair[p][1]];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      T s = 0;
#pragma unroll
      for (int p = 0; p < 6; ++p) s += m[kMomIdx.b3[k][p]] * q[p];
      b[3][k] = s;
    }
  }
  if (P >= 4) {
    T q[10];
#pragma unroll
    for (int t = 0; t < 10; ++t) q[t] = T(kTriMul[t]) * x[kTri[t][0]] * x[kTri[t][1]] * x[kTri[t][2]];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      T s = 0;
#pragma unroll
      for (int t = 0; t < 10; ++t) s += m[kMomIdx.b4[k][t]] * q[t];
      b[4][k] = s;
    }
  }
#pragma unroll
  for (int k = 1; k <= P; ++k) a[k] = x[0] * b[k][0] + x[1] * b[k][1] + x[2] * b[k][2];
  // Horner in phi
  T al = a[P];
#pragma unroll
  for (int k = P - 1; k >= 0; --k) al = a[k] + phi * al;
  al = al * phi;
  T be[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    T s = b[P][i];
#pragma unroll
    for (int k = P - 1; k >= 1; --k) s = b[k][i] + phi * s;
    be[i] = s * phi;
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) G[i] = c[i] * al + be[i];
}

// The far kernel's FP32 form of expansion<P>, accumulated into p.  Two
// identities shorten it:
//   a_k = x . b_k (k >= 1), so alpha = phi (M_0 + x . beta) needs no a_k, and
//   phi = 2 psi with psi = 1 / (|x-c|^2 + e_c),
// so with the record's moments scaled by 2^k (M'_k = 2^k M_k / (4 pi R)) and
// X = psi x the contractions nest:
//   h = M'_1 + X . (M'_2 + X . (M'_3 + X . M'_4)),  beta = psi h
//   alpha = psi (M'_0 + 2 X . h)
//   p += c alpha + psi h.
// cv = {c (3), e_c, M'_0..M'_P}.  78 vector instructions per target and cell at
// P = 4, none of which needs a product of coordinates kept in registers.
template <int P>
__device__ __forceinline__ void far_expansion_acc(const float* cv, const float x[3], float p[3]) {
  const float dx = x[0] - cv[0], dy = x[1] - cv[1], dz = x[2] - cv[2];
  const float psi = recip(fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, cv[3]))));
  const float* m = cv + 4;
  const float X[3] = {psi * x[0], psi * x[1], psi * x[2]};
  float t3[10], t2[6], h[3];
  if constexpr (P >= 3) {
#pragma unroll
    for (int i = 0; i < 10; ++i) {
      t3[i] = m[kMomOff[3] + i];
      if constexpr (P >= 4)
#pragma unroll
        for (int l = 0; l < 3; ++l)
          t3[i] = fmaf(X[l], m[kMomIdx.b4[l][i]], t3[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    t2[i] = m[kMomOff[2] + i];
    if constexpr (P >= 3)
#pragma unroll
      for (int l = 0; l < 3; ++l) t2[i] = fmaf(X[l], t3[kMomIdx.b3[l][i] - kMomOff[3]], t2[i]);
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    h[i] = m[1 + i];
#pragma unroll
    for (int l = 0; l < 3; ++l) h[i] = fmaf(X[l], t2[kMomIdx.b2[l][i] - kMomOff[2]], h[i]);
  }
  const float xh = fmaf(X[0], h[0], fmaf(X[1], h[1], X[2] * h[2]));
  const float alpha = psi * fmaf(2.f, xh, m[0]);
#pragma unroll
  for (int i = 0; i < 3; ++i) p[i] = fmaf(cv[i], alpha, fmaf(psi, h[i], p[i]));
}

#pragma clang fp contract(off)

__device__ __forceinline__ void project(double& x, double& y, double& z, double radius) {
  const double s = radius / sqrt(x * x + y * y + z * z);
  x = x * s;
  y = y * s;
  z = z * s;
}

// ---------------------------------------------------------------- binning
// Cell of each particle: the generator with the largest dot product (lowest
// index on ties); sort keys for targets (all particles) and sources (inactive
// particles get key ncell and sort last).
//
// The generators are fixed, so their search is laid out once: directions fall in
// 6 g x g bins (faces of the surrounding cube), and a bin lists, in ascending
// order, every generator that can be the nearest of a direction in it: those
// whose largest dot product over the bin is not below the largest of all the
// generators' smallest ones.  Bins of a quarter of a cell's width list 3-4 of
// them on average.  A bin with more than kBinMax, and a particle whose
// coordinates are no ordinary numbers, look through all generators.
// At 491,522 particles and 1,280 cells: 190 us over all generators, 13 in bins.
constexpr int kBinMax = 15;
struct LocBin {
  int count;  // -1: all generators
  int cell[kBinMax];
};

__host__ __device__ inline int loc_grid(int ncell) {
  int g = 4;
  while (g < 128 && 6 * g * g < 16 * ncell) g *= 2;
  return g;
}

// Bin of direction (px, py, pz), not all zero.
__device__ __forceinline__ int loc_bin(float px, float py, float pz, int g) {
  const float ax = fabsf(px), ay = fabsf(py), az = fabsf(pz);
  int face;
  float m, u, v;
  if (ax >= ay && ax >= az) {
    face = px >= 0.f ? 0 : 1, m = ax, u = py, v = pz;
  } else if (ay >= az) {
    face = py >= 0.f ? 2 : 3, m = ay, u = px, v = pz;
  } else {
    face = pz >= 0.f ? 4 : 5, m = az, u = px, v = py;
  }
  const float h = 0.5f * (float)g, q = h / m;
  const int iu = min(g - 1, max(0, (int)fmaf(u, q, h))), iv = min(g - 1, max(0, (int)fmaf(v, q, h)));
  return (face * g + iu) * g + iv;
}

__global__ __launch_bounds__(256) void ff_locate_bins(int ncell, int g, const lpm::Vec4<float>* __restrict__ gen,
                                                      LocBin* __restrict__ bins) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b >= 6 * g * g) return;
  const int face = b / (g * g), iu = b / g % g, iv = b % g;
  auto dir = [&](double u, double v, double d[3]) {
    const int ax = face >> 1;
    const double s = face & 1 ? -1.0 : 1.0, r = 1.0 / sqrt(1.0 + u * u + v * v);
    d[ax] = s * r;
    d[ax == 0 ? 1 : 0] = u * r;
    d[ax == 2 ? 1 : 2] = v * r;
  };
  const double w = 2.0 / g;
  double c[3], e[3];
  dir((iu + 0.5) * w - 1.0, (iv + 0.5) * w - 1.0, c);
  double half = 0.0;  // angular radius: the farthest corner, with room for the bin's own rounding
  for (int k = 0; k < 4; ++k) {
    dir((iu + (k & 1)) * w - 1.0, (iv + (k >> 1)) * w - 1.0, e);
    half = fmax(half, acos(fmin(1.0, c[0] * e[0] + c[1] * e[1] + c[2] * e[2])));
  }
  half += 1e-5;
  const double ch = cos(half), sh = sin(half);
  // of a generator at angle a (dot c, sine s): dot products over the bin lie in
  // [cos(a + half), cos(max(0, a - half))]; a zero generator has 0 everywhere
  auto bounds = [&](const lpm::Vec4<float>& q, double& lo, double& hi) {
    const double d = q.a * c[0] + q.b * c[1] + q.c * c[2];
    const double n2 = (double)q.a * q.a + (double)q.b * q.b + (double)q.c * q.c;
    const double s = sqrt(fmax(0.0, n2 - d * d)), n = sqrt(n2);
    lo = d <= -n * ch ? -n : d * ch - s * sh;
    hi = d >= n * ch ? n : d * ch + s * sh;
  };
  double floor_ = -1e300, lo, hi;
  for (int s = 0; s < ncell; ++s) {
    bounds(gen[s], lo, hi);
    floor_ = fmax(floor_, lo);
  }
  floor_ -= 1e-5;  // the FP32 products' rounding
  int count = 0;
  for (int s = 0; s < ncell; ++s) {
    bounds(gen[s], lo, hi);
    if (!(hi >= floor_)) continue;
    if (count >= kBinMax) {
      count = -1;
      break;
    }
    bins[b].cell[count++] = s;
  }
  bins[b].count = count;
}

__global__ __launch_bounds__(256) void ff_locate(int n, int ncell, int g, const lpm::Vec4<float>* __restrict__ gen,
                                                 const LocBin* __restrict__ bins, const double* __restrict__ x,
                                                 const double* __restrict__ y, const double* __restrict__ z,
                                                 const int* __restrict__ active, int* __restrict__ cellof,
                                                 lpm::CellSort sort) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float px = (float)x[i], py = (float)y[i], pz = (float)z[i];
  float best = -3.f;
  int bs = 0;
  auto visit = [&](const lpm::Vec4<float>& q, int s) {
    const float d = fmaf(q.a, px, fmaf(q.b, py, q.c * pz));
    if (d > best) {  // strict: the lowest index wins a tie
      best = d;
      bs = s;
    }
  };
  const float size = fabsf(px) + fabsf(py) + fabsf(pz);
  const LocBin* bin = nullptr;
  if (size > 1e-15f && size < 1e15f) {  // false for NaN
    bin = bins + loc_bin(px, py, pz, g);
    if (bin->count < 0) bin = nullptr;
  }
  if (bin) {
    const int count = bin->count;
    for (int k = 0; k < count; ++k) {
      const int s = bin->cell[k];
      visit(gen[s], s);
    }
  } else {
    for (int s = 0; s < ncell; ++s) visit(gen[s], s);
  }
  cellof[i] = bs;
  sort.tgt_key[i] = bs;
  sort.src_key[i] = active[i] ? bs : ncell;
  sort.tgt_val[i] = i;
  sort.src_val[i] = i;
}

// Start of every cell (and the end, index ncell) in the sorted key arrays: item i
// starts the cells after its predecessor's, up to its own.
__global__ __launch_bounds__(256) void ff_bounds(int n, int ncell, const unsigned* __restrict__ tkey,
                                                 const unsigned* __restrict__ skey, int* __restrict__ tgt_start,
                                                 int* __restrict__ src_start) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i > n) return;
  auto mark = [&](const unsigned* key, int* start) {
    const int prev = i > 0 ? (int)key[i - 1] : -1, cur = i < n ? (int)key[i] : ncell;
    for (int c = prev + 1; c <= cur; ++c) start[c] = i;
  };
  mark(tkey, tgt_start);
  mark(skey, src_start);
}

// Work items (cell, tile) for tiles of tileA and of tileB targets, in cell
// order; counts[0], counts[1] = their numbers.  One block of 1024 threads.
__global__ __launch_bounds__(1024) void ff_make_items(int ncell, const int* __restrict__ tgt_start, int tileA,
                                                      int tileB, int2* __restrict__ items_a,
                                                      int2* __restrict__ items_b, int* __restrict__ counts) {
  __shared__ int sa[1024], sb[1024];
  const int tid = threadIdx.x;
  const int per = (ncell + 1023) / 1024;
  const int c0 = min(ncell, tid * per), c1 = min(ncell, c0 + per);
  int na = 0, nb = 0;
  for (int c = c0; c < c1; ++c) {
    const int cnt = tgt_start[c + 1] - tgt_start[c];
    na += (cnt + tileA - 1) / tileA;
    nb += (cnt + tileB - 1) / tileB;
  }
  sa[tid] = na;
  sb[tid] = nb;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {  // inclusive scan
    const int va = tid >= off ? sa[tid - off] : 0, vb = tid >= off ? sb[tid - off] : 0;
    __syncthreads();
    sa[tid] += va;
    sb[tid] += vb;
    __syncthreads();
  }
  int oa = sa[tid] - na, ob = sb[tid] - nb;
  for (int c = c0; c < c1; ++c) {
    const int cnt = tgt_start[c + 1] - tgt_start[c];
    for (int j = 0; j * tileA < cnt; ++j) items_a[oa++] = make_int2(c, j);
    for (int j = 0; j * tileB < cnt; ++j) items_b[ob++] = make_int2(c, j);
  }
  if (tid == 1023) {
    counts[0] = sa[1023];
    counts[1] = sb[1023];
  }
}

// ---------------------------------------------------------------- packing
// Targets in cell order: FP32 {x, y, z, 0}.
__global__ __launch_bounds__(256) void ff_pack_targets(int n, const int* __restrict__ perm, const double* __restrict__ x,
                                                       const double* __restrict__ y, const double* __restrict__ z,
                                                       lpm::Vec4<float>* __restrict__ rec) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int p = perm[k];
  rec[k] = lpm::Vec4<float>{(float)x[p], (float)y[p], (float)z[p], 0.f};
}

// Per cell: FP64 centroids/radii of its sources and of its targets, the 10
// moments of w = zeta A about the source centroid, sum |w|; writes the far
// record (moments / (4 pi R)), the MLP record and FP64 geometry.
struct GeomArgs {
  int ncell;
  const int *src_perm, *src_start, *tgt_perm, *tgt_start;
  const double *x, *y, *z, *q, *area;
  double radius;
  float* far_rec;      // [ncell][40]: c(3), e_c, M0..M4 (35) / (4 pi R) with M0 scaled by 2 and Mk by 2^k, rho
  float* mlp_rec;      // [ncell][32]: c(3), 1/l, Q(9), s_out, pad(2), features 3..12, pad(6)
  const double* adir;  // [ncell][3] unit anchor direction of each cell's frame
  double* geo;         // [ncell][8]: src dir (3), src rho, tgt dir (3), tgt rho
  double* cen64;       // [ncell][3] FP64 source centroids
  double* mom64;       // [ncell][kNMom]
  double* pgeo;        // [npar][4]: the parents' source dir (3), rho
};

// Sums of K values over the block, in a fixed order, to every thread: eight values
// at a time through LDS, 32 lanes to a value.  `sh` holds kRedWords doubles.
constexpr int kRedWords = 8 * 256 + 48;
template <int K>
__device__ __forceinline__ void block_sums(double (&v)[K], double* sh) {
  double* res = sh + 8 * 256;
#pragma unroll
  for (int k0 = 0; k0 < K; k0 += 8) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (k0 + e < K) sh[e * 256 + threadIdx.x] = v[k0 + e];
    __syncthreads();
    const int e = threadIdx.x >> 5, l = threadIdx.x & 31;
    if (k0 + e < K) {
      double s = 0.0;
#pragma unroll
      for (int j = 0; j < 8; ++j) s += sh[e * 256 + l + 32 * j];
      for (int m = 16; m > 0; m >>= 1) s += __shfl_xor(s, m);
      if (l == 0) res[k0 + e] = s;
    }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = res[k];
}

// Cosine of the angle between (x, y, z) and a unit vector d for an angular radius; -1
// where either is not a number, so that the radius is pi and every pair near.
__device__ __forceinline__ double radius_cos(double x, double y, double z, double dx, double dy, double dz) {
  return fmax(-1.0, (x * dx + y * dy + z * dz) / sqrt(x * x + y * y + z * z));
}

// Smallest of a value over the block (no NaN), to every thread.
__device__ __forceinline__ double block_min(double v, double* sh) {
  for (int m = 32; m > 0; m >>= 1) v = fmin(v, __shfl_xor(v, m));
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  const double r = fmin(fmin(sh[0], sh[1]), fmin(sh[2], sh[3]));
  __syncthreads();
  return r;
}

// Area-weighted centroid c of the sources [s0, s1) (cell order), their
// moments M0..M4 of w = zeta A about c, sum |w| and angular radius about c's
// direction.  Every thread of the block gets the block's values.
struct SourceMoments {
  double cx, cy, cz, ux, uy, uz, rho, wabs;
  double m[kNMom];
};

// The centroid alone (v: area-weighted x, y, z and the area).
__device__ __forceinline__ void set_centroid(const double v[4], SourceMoments& r) {
  r.cx = v[3] > 0 ? v[0] / v[3] : 0.0;
  r.cy = v[3] > 0 ? v[1] / v[3] : 0.0;
  r.cz = v[3] > 0 ? v[2] / v[3] : 1.0;
  const double cn = sqrt(r.cx * r.cx + r.cy * r.cy + r.cz * r.cz);
  r.ux = r.cx / cn;
  r.uy = r.cy / cn;
  r.uz = r.cz / cn;
}

// Moments, sum |w| and angular radius about the centroid in r.  The radius is the
// arc cosine of the smallest cosine: one arc cosine a block, not one a source.
__device__ void source_moments(const GeomArgs& a, int s0, int s1, double* sh, SourceMoments& r) {
  double v[kNMom + 1];
#pragma unroll
  for (int k = 0; k <= kNMom; ++k) v[k] = 0.0;
  double cosmin = 1.0;
  for (int j = s0 + threadIdx.x; j < s1; j += 256) {
    const int p = a.src_perm[j];
    const double x = a.x[p], y = a.y[p], z = a.z[p];
    const double w = a.q[p] * a.area[p];
    const double d[3] = {x - r.cx, y - r.cy, z - r.cz};
    v[0] += w;
#pragma unroll
    for (int i = 0; i < 3; ++i) v[1 + i] += w * d[i];
#pragma unroll
    for (int i = 0; i < 6; ++i) v[kMomOff[2] + i] += w * d[kPair[i][0]] * d[kPair[i][1]];
#pragma unroll
    for (int i = 0; i < 10; ++i) v[kMomOff[3] + i] += w * d[kTri[i][0]] * d[kTri[i][1]] * d[kTri[i][2]];
#pragma unroll
    for (int i = 0; i < 15; ++i)
      v[kMomOff[4] + i] += w * d[kQuad[i][0]] * d[kQuad[i][1]] * d[kQuad[i][2]] * d[kQuad[i][3]];
    v[kNMom] += fabs(w);
    cosmin = fmin(cosmin, radius_cos(x, y, z, r.ux, r.uy, r.uz));
  }
  block_sums(v, sh);
#pragma unroll
  for (int k = 0; k < kNMom; ++k) r.m[k] = v[k];
  r.wabs = v[kNMom];
  r.rho = acos(block_min(cosmin, sh));
}

// The FP32 far record of far_expansion_acc: c, e_c = R^2 - |c|^2, the moments
// / (4 pi R) with M_0 and M_1 scaled by 2, M_2 by 4, M_3 by 8, M_4 by 16, rho.
__device__ void write_far_record(float* fr, const SourceMoments& sm, double R) {
  const double inv = 1.0 / (4.0 * kPi * R);
  fr[0] = (float)sm.cx;
  fr[1] = (float)sm.cy;
  fr[2] = (float)sm.cz;
  fr[3] = (float)(R * R - (sm.cx * sm.cx + sm.cy * sm.cy + sm.cz * sm.cz));
  for (int k = 0; k < kNMom; ++k)
    fr[4 + k] = (float)(sm.m[k] * inv * (k < 4 ? 2.0 : k < 10 ? 4.0 : k < 20 ? 8.0 : 16.0));
  fr[4 + kNMom] = (float)sm.rho;
}

// One block per cell, then one per parent.  Parent p is the four cells 4p .. 4p+3,
// whose sources are contiguous in cell order; it has a far record (after the
// cells' records) and its geometry only.  Both kinds wait on gathers and on the
// block's sums; at 491,522 particles and 1,280 + 320 blocks 36 us, against 88 + 42 with
// a sum of its own, nine barriers long, for each of the 45 values.
__global__ __launch_bounds__(256) void ff_cell_geometry(GeomArgs a) {
  __shared__ double sh[kRedWords];
  const bool cell = (int)blockIdx.x < a.ncell;
  const int c = cell ? blockIdx.x : blockIdx.x - a.ncell;
  const int s0 = a.src_start[cell ? c : 4 * c], s1 = a.src_start[cell ? c + 1 : 4 * c + 4];
  const int t0 = cell ? a.tgt_start[c] : 0, t1 = cell ? a.tgt_start[c + 1] : 0;
  double v[7] = {};
  for (int j = s0 + threadIdx.x; j < s1; j += 256) {
    const int p = a.src_perm[j];
    const double w = a.area[p];
    v[0] += w * a.x[p];
    v[1] += w * a.y[p];
    v[2] += w * a.z[p];
    v[3] += w;
  }
  for (int k = t0 + threadIdx.x; k < t1; k += 256) {
    const int p = a.tgt_perm[k];
    v[4] += a.x[p];
    v[5] += a.y[p];
    v[6] += a.z[p];
  }
  block_sums(v, sh);
  SourceMoments sm;
  set_centroid(v, sm);
  source_moments(a, s0, s1, sh, sm);
  if (!cell) {
    if (threadIdx.x == 0) {
      write_far_record(a.far_rec + (size_t)(a.ncell + c) * kCellRec, sm, a.radius);
      double* g = a.pgeo + (size_t)c * 4;
      g[0] = sm.ux;
      g[1] = sm.uy;
      g[2] = sm.uz;
      g[3] = sm.rho;
    }
    return;
  }
  const double cx = sm.cx, cy = sm.cy, cz = sm.cz, ux = sm.ux, uy = sm.uy, uz = sm.uz;
  const double* m = sm.m;
  const double wabs = sm.wabs, rho = sm.rho;
  // target cell direction and radius
  double tx = v[4], ty = v[5], tz = v[6];
  double tn = sqrt(tx * tx + ty * ty + tz * tz);
  if (!(tn > 0)) {
    tx = ux;
    ty = uy;
    tz = uz;
    tn = 1.0;
  }
  const double vx = tx / tn, vy = ty / tn, vz = tz / tn;
  double cosmin = 1.0;
  for (int k = t0 + threadIdx.x; k < t1; k += 256) {
    const int p = a.tgt_perm[k];
    const double x = a.x[p], y = a.y[p], z = a.z[p];
    cosmin = fmin(cosmin, radius_cos(x, y, z, vx, vy, vz));
  }
  const double trho = acos(block_min(cosmin, sh));
  if (threadIdx.x == 0) {
    const double R = a.radius;
    const double inv = 1.0 / (4.0 * kPi * R);
    write_far_record(a.far_rec + (size_t)c * kCellRec, sm, R);
    const double l = fmax(2.0 * R * sin(0.5 * rho), 1e-12);
    const double W = wabs + 1e-300;
    // cell frame: e3 = c/|c|, e1 = tangential part of (R anchor - c), e2 = e3 x e1
    double Q[3][3];
    Q[2][0] = ux;
    Q[2][1] = uy;
    Q[2][2] = uz;
    {
      const double* ad = a.adir + (size_t)c * 3;
      double ex = R * ad[0] - cx, ey = R * ad[1] - cy, ez = R * ad[2] - cz;
      const double dn = ex * ux + ey * uy + ez * uz;
      ex -= dn * ux;
      ey -= dn * uy;
      ez -= dn * uz;
      double en = sqrt(ex * ex + ey * ey + ez * ez);
      if (!(en > 1e-300)) {  // one-source cell: any tangent direction
        if (fabs(ux) < 0.9) {
          ex = 0.0; ey = -uz; ez = uy;
        } else {
          ex = uz; ey = 0.0; ez = -ux;
        }
        en = sqrt(ex * ex + ey * ey + ez * ez);
      }
      Q[0][0] = ex / en;
      Q[0][1] = ey / en;
      Q[0][2] = ez / en;
    }
    Q[1][0] = Q[2][1] * Q[0][2] - Q[2][2] * Q[0][1];
    Q[1][1] = Q[2][2] * Q[0][0] - Q[2][0] * Q[0][2];
    Q[1][2] = Q[2][0] * Q[0][1] - Q[2][1] * Q[0][0];
    const double S[3][3] = {{m[4], m[5], m[6]}, {m[5], m[7], m[8]}, {m[6], m[8], m[9]}};
    double QS[3][3];
    for (int i = 0; i < 3; ++i)
      for (int j = 0; j < 3; ++j) QS[i][j] = Q[i][0] * S[0][j] + Q[i][1] * S[1][j] + Q[i][2] * S[2][j];
    float* mr = a.mlp_rec + (size_t)c * kMlpRec;
    for (int k = 0; k < kMlpRec; ++k) mr[k] = 0.f;
    mr[0] = (float)cx;
    mr[1] = (float)cy;
    mr[2] = (float)cz;
    mr[3] = (float)(1.0 / l);
    for (int i = 0; i < 3; ++i)
      for (int j = 0; j < 3; ++j) mr[4 + 3 * i + j] = (float)Q[i][j];
    mr[13] = (float)(W * inv / (l * l));  // output scale s_out
    mr[16] = (float)(m[0] / W);
    for (int i = 0; i < 3; ++i) mr[17 + i] = (float)((Q[i][0] * m[1] + Q[i][1] * m[2] + Q[i][2] * m[3]) / (W * l));
    const int pr[6][2] = {{0, 0}, {0, 1}, {0, 2}, {1, 1}, {1, 2}, {2, 2}};
    for (int k = 0; k < 6; ++k) {
      const int i = pr[k][0], j = pr[k][1];
      mr[20 + k] = (float)((QS[i][0] * Q[j][0] + QS[i][1] * Q[j][1] + QS[i][2] * Q[j][2]) / (W * l * l));
    }
    double* g = a.geo + (size_t)c * 8;
    g[0] = ux;
    g[1] = uy;
    g[2] = uz;
    g[3] = rho;
    g[4] = vx;
    g[5] = vy;
    g[6] = vz;
    g[7] = trho;
    a.cen64[(size_t)c * 3 + 0] = cx;
    a.cen64[(size_t)c * 3 + 1] = cy;
    a.cen64[(size_t)c * 3 + 2] = cz;
    for (int k = 0; k < kNMom; ++k) a.mom64[(size_t)c * kNMom + k] = m[k];
  }
}

// Class of source cell s for target cell t (0 far, 1 band, 2 near) from
// their FP64 geometry rows (geo: src dir (3), src rho, tgt dir (3), tgt rho).
__device__ __forceinline__ int cell_class(const double* gt, const double* gs, double r_near, double r_band) {
  const double cosang = gt[4] * gs[0] + gt[5] * gs[1] + gt[6] * gs[2];
  const double ang = acos(fmin(1.0, fmax(-1.0, cosang)));
  const double pad = gt[7] + gs[3];
  return ang < r_near + pad ? 2 : (ang < r_band + pad ? 1 : 0);
}

// Per target cell t: class of every source cell (0 far, 1 band, 2 near) and
// compact lists of near and band cells.
struct ClassArgs {
  int ncell;
  const double* geo;
  double r_near, r_band;
  int* near_list;      // [ncell][ncell]
  int* near_count;
  int* band_list;      // [ncell][ncell]
  int* band_count;
};

__global__ __launch_bounds__(256) void ff_classify(ClassArgs a) {
  __shared__ int nn, nb;
  const int t = blockIdx.x;
  if (threadIdx.x == 0) {
    nn = 0;
    nb = 0;
  }
  __syncthreads();
  const double* gt = a.geo + (size_t)t * 8;
  for (int base = 0; base < a.ncell; base += 256) {
    const int s = base + threadIdx.x;
    int cls = -1;
    if (s < a.ncell) cls = cell_class(gt, a.geo + (size_t)s * 8, a.r_near, a.r_band);
    // ordered compaction: one wave at a time keeps lists sorted by s
    for (int w = 0; w < 4; ++w) {
      if ((int)(threadIdx.x >> 6) == w) {
        const unsigned long long mn = __ballot(cls == 2), mb = __ballot(cls == 1);
        const int lane = threadIdx.x & 63;
        const unsigned long long below = lane ? (~0ull >> (64 - lane)) : 0ull;
        if (cls == 2) a.near_list[(size_t)t * a.ncell + nn + __popcll(mn & below)] = s;
        if (cls == 1) a.band_list[(size_t)t * a.ncell + nb + __popcll(mb & below)] = s;
        if (lane == 0) {
          nn += __popcll(mn);
          nb += __popcll(mb);
        }
      }
      __syncthreads();
    }
  }
  if (threadIdx.x == 0) {
    a.near_count[t] = nn;
    a.band_count[t] = nb;
  }
}

// Per target cell t: the far kernel's list of expansion records, in order.
// Cells are visited in groups (4 siblings with the coarse level, else 1); a
// group of 4 far cells whose parent p is far enough, angle >= r_par + rho_t +
// rho_p, contributes the parent's record ncell + p, else every one of its
// cells that is not near contributes its own.
struct FarListArgs {
  int ncell, group;  // group 4 (coarse level) or 1
  const double* geo;
  const double* pgeo;
  double r_near, r_band, r_par;
  int* far_list;   // [ncell][ncell]
  int* far_count;
};

__global__ __launch_bounds__(256) void ff_far_list(FarListArgs a) {
  __shared__ int sc[256];
  __shared__ int base;
  const int t = blockIdx.x;
  const double* gt = a.geo + (size_t)t * 8;
  if (threadIdx.x == 0) base = 0;
  const int ng = a.ncell / a.group;
  for (int g0 = 0; g0 < ng; g0 += 256) {
    const int g = g0 + threadIdx.x;
    int ent[4];
    int n = 0;
    if (g < ng) {
      int cls[4];
      bool all_far = true;
      for (int k = 0; k < a.group; ++k) {
        cls[k] = cell_class(gt, a.geo + (size_t)(g * a.group + k) * 8, a.r_near, a.r_band);
        all_far = all_far && cls[k] == 0;
      }
      bool parent = false;
      if (a.group == 4 && all_far) {
        const double* gp = a.pgeo + (size_t)g * 4;
        const double cosang = gt[4] * gp[0] + gt[5] * gp[1] + gt[6] * gp[2];
        parent = acos(fmin(1.0, fmax(-1.0, cosang))) >= a.r_par + gt[7] + gp[3];
      }
      if (parent) {
        ent[n++] = a.ncell + g;
      } else {
        for (int k = 0; k < a.group; ++k)
          if (cls[k] != 2) ent[n++] = g * a.group + k;
      }
    }
    // ordered placement: inclusive scan of the counts over the block
    sc[threadIdx.x] = n;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {
      const int v = threadIdx.x >= (unsigned)d ? sc[threadIdx.x - d] : 0;
      __syncthreads();
      sc[threadIdx.x] += v;
      __syncthreads();
    }
    int* out = a.far_list + (size_t)t * a.ncell + base + sc[threadIdx.x] - n;
    for (int i = 0; i < n; ++i) out[i] = ent[i];
    __syncthreads();
    if (threadIdx.x == 255) base += sc[255];
    __syncthreads();
  }
  if (threadIdx.x == 0) a.far_count[t] = base;
}

// --------------------------------------------------------- near field
struct NearArgs {
  const lpm::Vec4<float>* tgt;  // cell-ordered targets
  const int* tgt_perm;          // particle index of each ordered target
  const int* tgt_start;
  const float* src;             // cell-ordered source records (SREC)
  const int* src_start;
  const int* near_list;
  const int* near_count;
  const int2* items;            // (target cell, wave tile)
  const int* n_items;  // device count
  int ncell;
  double* out;                  // [split][3][nt] FP64, cell order
  int nt;
  int nsplit;                   // near lists are split in nsplit parts (grid y)
};

// Targets [k0, k0 + 64 R) of cell t.
template <int R>
__device__ __forceinline__ void near_item(const NearArgs& a, int t, int k0, int k_end) {
  using P = lpm::SphereBS<float, false>;
  const int lane = threadIdx.x & 63;
  lpm::Vec4<float> tv[R];
  int tid[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int k = k0 + 64 * r + lane;
    const int kc = k < k_end ? k : k_end - 1;
    tv[r] = a.tgt[kc];
    tid[r] = k < k_end ? a.tgt_perm[kc] : -1;
  }
  float S[R][3], C[R][3];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) S[r][c] = C[r][c] = 0.f;
  // this split's share of the near list
  const int nn = a.near_count[t];
  const int split = blockIdx.y;
  const int qb = (int)((long long)nn * split / a.nsplit), qe = (int)((long long)nn * (split + 1) / a.nsplit);
  double* out = a.out + (size_t)split * 3 * a.nt;
  // particle ids of the wave's targets: ascending inside a cell (stable binning)
  const int id_lo = a.tgt_perm[k0], id_hi = a.tgt_perm[min(k0 + 64 * R, k_end) - 1];
  for (int q = qb; q < qe; ++q) {
    const int s = __builtin_amdgcn_readfirstlane(a.near_list[(size_t)t * a.ncell + q]);
    const int j0 = a.src_start[s], j1 = a.src_start[s + 1];
    for (int jt = j0; jt < j1; jt += kKT) {
      const int je = min(j1, jt + kKT);
      // a target's own source lives in its own cell, in the source tile whose
      // (ascending) particle ids span the target's
      const bool checked = s == t && __float_as_int(a.src[(size_t)jt * lpm::SREC + P::IDX]) <= id_hi &&
                           __float_as_int(a.src[(size_t)(je - 1) * lpm::SREC + P::IDX]) >= id_lo;
      float p[R][3];
#pragma unroll
      for (int r = 0; r < R; ++r) p[r][0] = p[r][1] = p[r][2] = 0.f;
      if (!checked) {
        // each source's record is loaded one source ahead of its arithmetic, as
        // in the plain pair kernel
        float sv[lpm::SREC];
#pragma unroll
        for (int e = 0; e < lpm::SREC; ++e) sv[e] = a.src[(size_t)jt * lpm::SREC + e];
#pragma unroll 2
        for (int j = jt; j < je; ++j) {
          const int jn = j + 1 < je ? j + 1 : j;
          float sn[lpm::SREC];
#pragma unroll
          for (int e = 0; e < lpm::SREC; ++e) sn[e] = a.src[(size_t)jn * lpm::SREC + e];
          lpm::W4<float> w[R];
          float f[R];
#pragma unroll
          for (int r = 0; r < R; ++r) P::arg(tv[r], sv, w[r]);
#pragma unroll
          for (int r = 0; r < R; ++r) f[r] = P::trans(w[r]);
#pragma unroll
          for (int r = 0; r < R; ++r) P::acc(sv, w[r], f[r], p[r]);
#pragma unroll
          for (int e = 0; e < lpm::SREC; ++e) sv[e] = sn[e];
        }
      } else {
        for (int j = jt; j < je; ++j) {
          const float* sr = a.src + (size_t)j * lpm::SREC;
          float sv[lpm::SREC];
#pragma unroll
          for (int e = 0; e < lpm::SREC; ++e) sv[e] = sr[e];
          const int sidx = __float_as_int(sv[P::IDX]);
#pragma unroll
          for (int r = 0; r < R; ++r) {
            lpm::W4<float> w;
            P::arg(tv[r], sv, w);
            const float f = P::trans(w);
            float tmp[3] = {0.f, 0.f, 0.f};
            P::acc(sv, w, f, tmp);
            const bool self = sidx == tid[r];
#pragma unroll
            for (int c = 0; c < 3; ++c) p[r][c] += self ? 0.f : tmp[c];
          }
        }
      }
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) lpm::two_sum_acc(S[r][c], C[r][c], p[r][c]);
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int k = k0 + 64 * r + lane;
    if (k < k_end)
#pragma unroll
      for (int c = 0; c < 3; ++c) out[(size_t)c * a.nt + k] = (double)S[r][c] + (double)C[r][c];
  }
}

// A cell's last tile takes one target a lane where that holds it: for cells of 24
// targets (level 5) the expansions take 73 us instead of 128, the near sums 23 instead
// of 27 and an evaluation 665 instead of 708; at 384 a cell both gain 2 %.
__global__ __launch_bounds__(256) void ff_near_kernel(NearArgs a) {
  // the wave's item index is wave-uniform: readfirstlane puts it (and every
  // index and record address derived from it) in scalar registers
  const int item = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (item >= *a.n_items) return;
  const int2 it = a.items[item];
  const int t = it.x;
  const int k0 = a.tgt_start[t] + it.y * 64 * kR;
  const int k_end = a.tgt_start[t + 1];
  if (k_end - k0 > 64)
    near_item<kR>(a, t, k0, k_end);
  else
    near_item<1>(a, t, k0, k_end);
}

// ------------------------------------------------------- far (expansion)
// Every record of a target cell's far list (cells not near it, or their
// parents) by its expansion.  The list is split in gridDim.y contiguous
// ranges, one FP64 partial per range, so that the launch has several rounds
// of waves and its last round is short.
struct FarArgs {
  const lpm::Vec4<float>* tgt;
  const int* tgt_start;
  const float* cell;          // far records: cells, then parents
  const int* far_list;        // [ncell][ncell] record indices per target cell
  const int* far_count;
  const int2* items;
  const int* n_items;  // device count
  int ncell, nt;
  double* part;               // [gridDim.y][3][nt] this launch's partials
};

// Records pass through LDS, kFarBatch at a time and per wave, to vector registers: a
// vector instruction with a scalar operand takes 4.2 cycles, one without 2.9, and
// each of a record's words is an operand of kR targets.  At 491,522 targets and some
// 460 records each (P = 4): 411 us, against 532 with scalar records and the
// products of coordinates in registers; 467 at 3 and 4 targets a lane, whose tiles
// leave more of a cell's last one empty, 443 at 4 waves a SIMD.  (The near sums take
// 8 words a source for 11 instructions: there the LDS reads cost what they save,
// 863 against 815 us.)
constexpr int kRec4 = kCellRec / 4;
constexpr int kFarBatch = 64 / kRec4;  // a 16-byte word a lane

template <int P, int R>
__device__ __forceinline__ void far_item(const FarArgs& a, int t, int k0, int k_end, float4 (*stage)[kFarBatch * kRec4]) {
  const int lane = threadIdx.x & 63;
  float X[R][3];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int k = k0 + 64 * r + lane;
    const lpm::Vec4<float> v = a.tgt[k < k_end ? k : k_end - 1];
    X[r][0] = v.a;
    X[r][1] = v.b;
    X[r][2] = v.c;
  }
  float S[R][3], C[R][3];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) S[r][c] = C[r][c] = 0.f;
  const int* list = a.far_list + (size_t)t * a.ncell;
  const int cnt = a.far_count[t];
  const int q_lo = (int)((long long)cnt * blockIdx.y / gridDim.y);
  const int q_hi = (int)((long long)cnt * (blockIdx.y + 1) / gridDim.y);
  // a lane fetches one 16-byte word of the batch; past the end of the list the last
  // record's again
  const float4* cell4 = reinterpret_cast<const float4*>(a.cell);
  float4 next;
  auto fetch = [&](int q) {
    next = cell4[(size_t)list[min(q + lane / kRec4, q_hi - 1)] * kRec4 + lane % kRec4];
  };
  float p[R][3];
#pragma unroll
  for (int r = 0; r < R; ++r) p[r][0] = p[r][1] = p[r][2] = 0.f;
  if (q_lo < q_hi) fetch(q_lo);
  int buf = 0, done = 0;
  for (int q = q_lo; q < q_hi; q += kFarBatch, buf ^= 1) {
    float4* st = stage[buf];
    if (lane < kFarBatch * kRec4) st[lane] = next;
    __builtin_amdgcn_wave_barrier();  // LDS serves a wave's accesses in order
    if (q + kFarBatch < q_hi) fetch(q + kFarBatch);
    const int n = min(kFarBatch, q_hi - q);
    for (int e = 0; e < n; ++e) {
      constexpr int NV = 4 + kMomOff[P] + (P + 1) * (P + 2) / 2;  // c, e_c, M'0..M'P
      float cv[(NV + 3) / 4 * 4];
#pragma unroll
      for (int w = 0; w < (NV + 3) / 4; ++w) {
        const float4 v = st[e * kRec4 + w];
        cv[4 * w] = v.x, cv[4 * w + 1] = v.y, cv[4 * w + 2] = v.z, cv[4 * w + 3] = v.w;
      }
#pragma unroll
      for (int r = 0; r < R; ++r) far_expansion_acc<P>(cv, X[r], p[r]);
    }
    // one compensated block per 10 batches of this part of the list
    if (++done == 10 || q + kFarBatch >= q_hi) {
      done = 0;
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          lpm::two_sum_acc(S[r][c], C[r][c], p[r][c]);
          p[r][c] = 0.f;
        }
    }
  }
  double* out = a.part + (size_t)blockIdx.y * 3 * a.nt;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int k = k0 + 64 * r + lane;
    if (k < k_end)
#pragma unroll
      for (int c = 0; c < 3; ++c) out[(size_t)c * a.nt + k] = (double)S[r][c] + (double)C[r][c];
  }
}

template <int P>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void ff_far_kernel(FarArgs a) {
  __shared__ float4 stage[4][2][kFarBatch * kRec4];
  // the wave's item index is wave-uniform: readfirstlane puts it (and every
  // index derived from it) in scalar registers
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int item = blockIdx.x * 4 + wid;
  if (item >= *a.n_items) return;
  const int2 it = a.items[item];
  const int t = it.x;
  const int k0 = a.tgt_start[t] + it.y * 64 * kR;
  const int k_end = a.tgt_start[t + 1];
  if (k_end - k0 > 64)
    far_item<P, kR>(a, t, k0, k_end, stage[wid]);
  else
    far_item<P, 1>(a, t, k0, k_end, stage[wid]);
}

// --------------------------------------------------- MLP correction (MFMA)
// Target position in the cell frame, Q (x - c) / l.
__device__ __forceinline__ void mlp_local(const float* mr, float x, float y, float z, float loc[3]) {
  const float dx = (x - mr[0]) * mr[3], dy = (y - mr[1]) * mr[3], dz = (z - mr[2]) * mr[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) loc[i] = fmaf(mr[4 + 3 * i], dx, fmaf(mr[5 + 3 * i], dy, mr[6 + 3 * i] * dz));
}

// Input f of a sample: 0..2 the local position, 3..12 the cell's moment features.
__device__ __forceinline__ float mlp_feature(const float* mr, const float loc[3], int f) {
  if (f < 3) return loc[f];
  if (f < 13) return mr[16 + (f - 3)];
  return 0.f;
}

// r^(P+2) for squared radius r2 and expansion order P in 2..4
__device__ __forceinline__ float out_pow(float r2, int order) {
  const float r4 = r2 * r2;
  return order == 2 ? r4 : (order == 3 ? r4 * sqrtf(r2) : r4 * r2);
}

// s_out / r^(P+2) for the local position
__device__ __forceinline__ float mlp_out_scale(const float* mr, const float loc[3], int order) {
  const float r2 = fmaf(loc[0], loc[0], fmaf(loc[1], loc[1], loc[2] * loc[2]));
  return mr[13] * __builtin_amdgcn_rcpf(out_pow(r2, order));
}

struct MlpCorrArgs {
  const lpm::Vec4<float>* tgt;
  const int* tgt_start;
  const float* mlp_rec;
  const int* band_list;
  const int* band_count;
  const int2* items;  // (target cell, 64-target tile)
  const int* n_items;  // device count
  int ncell, nt, order;
  const lpm::mlp_t* frag;
  const float* bias;
  double* part;       // [3][nt] this launch's partial
};

// 512 threads: 8 waves (2 per SIMD) share one LDS copy of the weights, which
// alone takes half a CU's LDS.
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void ff_mlp_kernel(MlpCorrArgs a) {
  __shared__ __attribute__((aligned(16))) lpm::mlp_t sfrag[lpm::kMlpFragElems];
  __shared__ __attribute__((aligned(16))) float sbias[lpm::kMlpBiasElems];
  for (int t = threadIdx.x; t < lpm::kMlpFragElems / 8; t += blockDim.x)
    reinterpret_cast<lpm::mlpx8_t*>(sfrag)[t] = reinterpret_cast<const lpm::mlpx8_t*>(a.frag)[t];
  for (int t = threadIdx.x; t < lpm::kMlpBiasElems; t += blockDim.x) sbias[t] = a.bias[t];
  __syncthreads();
  constexpr int NCT = kMlpNct;
  const int lane = threadIdx.x & 63, g = lane >> 4;
  const int waves = gridDim.x * (blockDim.x >> 6);
  const int n_items = *a.n_items;
  const int wave0 = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
  for (int item = wave0; item < n_items; item += waves) {
    const int2 it = a.items[item];
    const int t = it.x;
    const int k0 = a.tgt_start[t] + it.y * kMlpTile;
    const int k_end = a.tgt_start[t + 1];
    float xs[NCT][3];
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
      const int k = min(k0 + 16 * ct + (lane & 15), k_end - 1);
      const lpm::Vec4<float> v = a.tgt[k];
      xs[ct][0] = v.a;
      xs[ct][1] = v.b;
      xs[ct][2] = v.c;
    }
    float acc[NCT][3];
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) acc[ct][0] = acc[ct][1] = acc[ct][2] = 0.f;
    const int nb = a.band_count[t];
    for (int q = 0; q < nb; ++q) {
      const int s = __builtin_amdgcn_readfirstlane(a.band_list[(size_t)t * a.ncell + q]);
      const float* mr = a.mlp_rec + (size_t)s * kMlpRec;
      // the cell's 10 moment features (scalar loads); lane group g holds inputs
      // 8g .. 8g+7: g = 0 the local position and features 3..7, g = 1 features
      // 8..12, g = 2, 3 the zero padding -- selected without branches
      float mv[10];
#pragma unroll
      for (int k = 0; k < 10; ++k) mv[k] = mr[16 + k];
      lpm::mlpx8_t in8[NCT];
      float loc[NCT][3];
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        mlp_local(mr, xs[ct][0], xs[ct][1], xs[ct][2], loc[ct]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float f0 = e < 3 ? loc[ct][e] : mv[e - 3];
          const float f1 = e < 5 ? mv[5 + e] : 0.f;
          in8[ct][e] = (lpm::mlp_t)(g == 0 ? f0 : (g == 1 ? f1 : 0.f));
        }
      }
      float o[NCT][4];
      lpm::mlp_wave_forward<NCT, lpm::kActIsru>(in8, sfrag, sbias, o);
      // lanes 0..15 hold the outputs: scale, rotate to world axes (Q^T o), accumulate
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        const float so = mlp_out_scale(mr, loc[ct], a.order);
        const float o0 = o[ct][0] * so, o1 = o[ct][1] * so, o2 = o[ct][2] * so;
#pragma unroll
        for (int c = 0; c < 3; ++c) acc[ct][c] = fmaf(mr[4 + c], o0, fmaf(mr[7 + c], o1, fmaf(mr[10 + c], o2, acc[ct][c])));
      }
    }
    if (g == 0) {
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        const int k = k0 + 16 * ct + lane;
        if (k < k_end)
#pragma unroll
          for (int c = 0; c < 3; ++c) a.part[(size_t)c * a.nt + k] = (double)acc[ct][c];
      }
    }
  }
}

// ---------------------------------------------------------------- epilogue
// V = the near partials, the far partials, then the network's, summed in this
// fixed order; u = V x x, in the particles' own order.
__global__ __launch_bounds__(256) void ff_epilogue(int nt, int nparts, const int* __restrict__ perm,
                                                   const double* __restrict__ part, const double* __restrict__ x,
                                                   const double* __restrict__ y, const double* __restrict__ z,
                                                   double* __restrict__ u, double* __restrict__ v,
                                                   double* __restrict__ w) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nt) return;
  const int p = perm[k];
  double V[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) V[c] = part[(size_t)c * nt + k];
  for (int sp = 1; sp < nparts; ++sp)
#pragma unroll
    for (int c = 0; c < 3; ++c) V[c] += part[(size_t)(3 * sp + c) * nt + k];
  const double A0 = V[0], A1 = V[1], A2 = V[2];
  const double px = x[p], py = y[p], pz = z[p];
  u[p] = A1 * pz - A2 * py;
  v[p] = A2 * px - A0 * pz;
  w[p] = A0 * py - A1 * px;
}

// --------------------------------------------------- training samples
// Sample q: a random target (particle) and a random band cell of its cell.
// Inputs: the 13 MLP features; target: Q (G_exact - G_expansion) / (4 pi R) r^(P+2) / s_out,
// the remainder in the cell frame and scaled, in FP64 (G_exact over the cell's
// sources, with w = zeta A).  ids receives (particle, cell) of each sample.
struct SampleArgs {
  int n_samples;
  unsigned long long seed;
  int nt, ncell, order;
  const int* tgt_perm;
  const unsigned* tgt_cell;
  const int *src_perm, *src_start, *band_list, *band_count;
  const double *x, *y, *z, *q, *area;
  const double *cen64, *mom64;
  const float* mlp_rec;
  double radius;
  float* X;  // [n][13]
  float* Y;  // [n][3]
  int* ids;  // [n][2]: target particle, source cell (-1, -1 for an invalid sample)
  int draws = 1;  // band cells drawn per sample; the one nearest the target is kept
};

__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

__device__ void expansion_fp64(int order, const double* c, const double* m, double R, const double x[3],
                               double G[3]) {
  const double e_c = R * R - (c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
  if (order == 2) expansion<2, double>(c, e_c, m, x, G);
  else if (order == 3) expansion<3, double>(c, e_c, m, x, G);
  else expansion<4, double>(c, e_c, m, x, G);
}

__global__ __launch_bounds__(256) void ff_make_samples(SampleArgs a) {
  const int qi = blockIdx.x * blockDim.x + threadIdx.x;
  if (qi >= a.n_samples) return;
  unsigned long long h = mix64(a.seed ^ mix64((unsigned long long)qi));
  int ok = 0, pid = -1, sid = -1;
  float feat[13];
  float tgt3[3] = {0.f, 0.f, 0.f};
  for (int attempt = 0; attempt < 8 && !ok; ++attempt) {
    const int k = (int)(h % (unsigned long long)a.nt);
    h = mix64(h);
    const int t = (int)a.tgt_cell[k];
    const int nb = a.band_count[t];
    if (nb == 0) continue;
    const int p = a.tgt_perm[k];
    const double x = a.x[p], y = a.y[p], z = a.z[p];
    // band cell: the nearest (centroid distance) of `draws` uniform draws, so
    // that the cells whose remainders dominate the error are sampled more
    int s = -1;
    double best = 0.0;
    for (int d = 0; d < a.draws; ++d) {
      const int c = a.band_list[(size_t)t * a.ncell + (int)(h % (unsigned long long)nb)];
      h = mix64(h);
      const double* cc = a.cen64 + (size_t)c * 3;
      const double d2 = (x - cc[0]) * (x - cc[0]) + (y - cc[1]) * (y - cc[1]) + (z - cc[2]) * (z - cc[2]);
      if (s < 0 || d2 < best) {
        s = c;
        best = d2;
      }
    }
    const double R = a.radius;
    double Ge[3] = {0.0, 0.0, 0.0};
    for (int j = a.src_start[s]; j < a.src_start[s + 1]; ++j) {
      const int pj = a.src_perm[j];
      const double dx = x - a.x[pj], dy = y - a.y[pj], dz = z - a.z[pj];
      const double D = 0.5 * (dx * dx + dy * dy + dz * dz +
                              (R * R - (a.x[pj] * a.x[pj] + a.y[pj] * a.y[pj] + a.z[pj] * a.z[pj])));
      const double w = a.q[pj] * a.area[pj] / D;
      Ge[0] += w * a.x[pj];
      Ge[1] += w * a.y[pj];
      Ge[2] += w * a.z[pj];
    }
    double Gm[3];
    const double* c64 = a.cen64 + (size_t)s * 3;
    const double xv[3] = {x, y, z};
    expansion_fp64(a.order, c64, a.mom64 + (size_t)s * kNMom, R, xv, Gm);
    const float* mr = a.mlp_rec + (size_t)s * kMlpRec;
    // local position in FP64 for the scaling, FP32 (as at inference) for the inputs
    const double il = (double)mr[3];
    double r2 = 0.0;
    for (int i = 0; i < 3; ++i) {
      const double li = ((double)mr[4 + 3 * i] * (x - c64[0]) + (double)mr[5 + 3 * i] * (y - c64[1]) +
                         (double)mr[6 + 3 * i] * (z - c64[2])) * il;
      r2 += li * li;
    }
    const double rp = a.order == 2 ? r2 * r2 : (a.order == 3 ? r2 * r2 * sqrt(r2) : r2 * r2 * r2);
    const double inv = rp / (4.0 * kPi * R) / (double)mr[13];
    for (int i = 0; i < 3; ++i)
      tgt3[i] = (float)(((double)mr[4 + 3 * i] * (Ge[0] - Gm[0]) + (double)mr[5 + 3 * i] * (Ge[1] - Gm[1]) +
                         (double)mr[6 + 3 * i] * (Ge[2] - Gm[2])) * inv);
    float loc[3];
    mlp_local(mr, (float)x, (float)y, (float)z, loc);
    for (int f = 0; f < 13; ++f) feat[f] = mlp_feature(mr, loc, f);
    ok = 1;
    pid = p;
    sid = s;
  }
  for (int f = 0; f < 13; ++f) a.X[(size_t)qi * 13 + f] = ok ? feat[f] : 0.f;
  for (int c = 0; c < 3; ++c) a.Y[(size_t)qi * 3 + c] = tgt3[c];
  a.ids[(size_t)qi * 2] = pid;
  a.ids[(size_t)qi * 2 + 1] = sid;
}

// ---------------------------------------------------------- RK4 algebra
__global__ __launch_bounds__(256) void ff_stage(int n, double dt, double omega, double radius, double h, int first,
                                                int make_input, const double* __restrict__ x,
                                                const double* __restrict__ y, const double* __restrict__ z,
                                                const double* __restrict__ q, const double* __restrict__ u,
                                                const double* __restrict__ v, const double* __restrict__ w,
                                                double* kx, double* ky, double* kz, double* kq, double* xi,
                                                double* yi, double* zi, double* qi) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double vx = first ? u[i] : kx[i], vy = first ? v[i] : ky[i], vz = first ? w[i] : kz[i];
  const double dq = -dt * 2.0 * omega * vz / radius;
  const double a = dt * vx, b = dt * vy, c = dt * vz;
  kx[i] = a;
  ky[i] = b;
  kz[i] = c;
  kq[i] = dq;
  if (make_input) {
    double px = x[i] + h * a, py = y[i] + h * b, pz = z[i] + h * c;
    project(px, py, pz, radius);
    xi[i] = px;
    yi[i] = py;
    zi[i] = pz;
    qi[i] = q[i] + h * dq;
  }
}

__global__ __launch_bounds__(256) void ff_combine(int n, double radius, double* x, double* y, double* z, double* q,
                                                  const double* const* __restrict__ k) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double* st[4] = {x, y, z, q};
  double v[4];
  for (int c = 0; c < 4; ++c)
    v[c] = st[c][i] + k[c * 4 + 0][i] / 6.0 + k[c * 4 + 1][i] / 3.0 + k[c * 4 + 2][i] / 3.0 + k[c * 4 + 3][i] / 6.0;
  project(v[0], v[1], v[2], radius);
  for (int c = 0; c < 4; ++c) st[c][i] = v[c];
}

__global__ __launch_bounds__(256) void ff_project(int n, double radius, double* x, double* y, double* z) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double a = x[i], b = y[i], c = z[i];
  project(a, b, c, radius);
  x[i] = a;
  y[i] = b;
  z[i] = c;
}

// max_i |a_i - b_i| and max_i |b_i| over 3-vectors (two-pass, deterministic)
__global__ __launch_bounds__(256) void ff_err_partial(int n, const double* __restrict__ au, const double* __restrict__ av,
                                                      const double* __restrict__ aw, const double* __restrict__ bu,
                                                      const double* __restrict__ bv, const double* __restrict__ bw,
                                                      double* __restrict__ part) {
  __shared__ double s0[256], s1[256];
  double d = 0.0, m = 0.0;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const double ex = au[i] - bu[i], ey = av[i] - bv[i], ez = aw[i] - bw[i];
    d = fmax(d, sqrt(ex * ex + ey * ey + ez * ez));
    m = fmax(m, sqrt(bu[i] * bu[i] + bv[i] * bv[i] + bw[i] * bw[i]));
  }
  s0[threadIdx.x] = d;
  s1[threadIdx.x] = m;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) {
      s0[threadIdx.x] = fmax(s0[threadIdx.x], s0[threadIdx.x + k]);
      s1[threadIdx.x] = fmax(s1[threadIdx.x], s1[threadIdx.x + k]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s0[0];
    part[2 * blockIdx.x + 1] = s1[0];
  }
}

}  // namespace

// ====================================================================== object
struct lpm_bve_ff {
  lpm_ctx* ctx = nullptr;
  int n = 0, ns = 0, ncell = 0;
  double radius = 1.0, omega = 0.0, r_near = 0.1, r_band = 0.45;
  int order = 4;  // expansion order of far cells
  int draws = 1;  // training samples: band cells drawn per sample (nearest kept)
  DevBuf x, y, z, q, u, v, w, area;
  DevBuf k[4][4];
  DevBuf xi, yi, zi, qi;
  DevBuf pu, pv, pw;  // plain-sum velocity (judge)
  // binning: cell-ordered particle lists rebuilt at every evaluation
  DevBuf src_perm, src_start, tgt_perm, tgt_start;
  DevBuf cellof, active, sort_tmp, item_count;
  const unsigned* tgt_cell = nullptr;  // cell of each ordered target, in sort_tmp
  DevBuf gen, adir;  // cell generator directions (float4), frame anchor directions (FP64)
  DevBuf bins;       // LocBin per direction bin: the generators' search, laid out once
  DevBuf trec, srec, far_rec, mlp_rec, geo, cen64, mom64;
  DevBuf near_list, near_count, band_list, band_count;
  DevBuf far_list, far_count;  // expansion records per target cell (cells or parents)
  DevBuf pgeo;                 // coarse level: parent geometry [ncell / 4][4]
  int npar = 0;                // parents in use (0: no coarse level)
  double r_par = 0.0;          // a parent replaces its 4 cells beyond this radius
  DevBuf items, mlp_items;
  DevBuf Vpart;        // FP64 partials [near_split + far_split + 1][3][n]: near, far, network
  int near_split = 1;  // near lists split in this many parts (fills the chip)
  int far_split = 1;   // far cells split in this many ranges
  DevBuf list_plain;  // ascending active list for the plain path
  DevBuf tgt_plain, src_plain, partial_plain;
  DevBuf ptrs, err_part;
  DevBuf sx, sy, sid;  // collected training set: inputs, targets, (particle, cell)
  int n_items = 0, n_mlp_items = 0;
  int64_t n_collected = 0, cap_collected = 0;
  lpm::Mlp net;
  bool trained = false;
  double ys = 0.0;  // RMS of the training targets (0: not fixed yet)
  int online_n = 0, online_epochs = 1, online_batch = 4096, online_rounds = 0;
  double online_from = 0.0;  // fine-tune only at judged errors above online_from * tol
  double online_lr = 2e-4;
  bool loaded = false;  // false after a failed particle reload
};

namespace {

int ff_upload(lpm_ctx* ctx, DevBuf& b, const void* host, size_t bytes) {
  LPM_HIP(ctx, b.ensure(bytes));
  if (host && bytes) LPM_HIP(ctx, hipMemcpyAsync(b.p, host, bytes, hipMemcpyHostToDevice, ctx->stream));
  return LPM_OK;
}

// Bin the particles at (x, y, z) into cells: cell-ordered target and source
// lists (stable: ascending particle index inside a cell), cell starts, items.
int ff_bin(lpm_bve_ff* f, const double* x, const double* y, const double* z) {
  lpm_ctx* ctx = f->ctx;
  const int n = f->n, nc = f->ncell;
  const lpm::CellSort sort = lpm::cell_sort_input(f->sort_tmp, n);
  hipLaunchKernelGGL(ff_locate, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, n, nc, loc_grid(nc),
                     f->gen.as<lpm::Vec4<float>>(), f->bins.as<LocBin>(), x, y, z, f->active.as<int>(),
                     f->cellof.as<int>(), sort);
  const unsigned* src_key = nullptr;
  lpm::cell_sort(ctx->stream, f->sort_tmp, n, 32 - __builtin_clz((unsigned)nc), f->tgt_perm.as<int>(),
                 f->src_perm.as<int>(), &f->tgt_cell, &src_key);  // keys 0..ncell
  hipLaunchKernelGGL(ff_bounds, dim3((n + 1 + 255) / 256), dim3(256), 0, ctx->stream, n, nc, f->tgt_cell, src_key,
                     f->tgt_start.as<int>(), f->src_start.as<int>());
  hipLaunchKernelGGL(ff_make_items, dim3(1), dim3(1024), 0, ctx->stream, nc, f->tgt_start.as<int>(), 64 * kR, kMlpTile,
                     f->items.as<int2>(), f->mlp_items.as<int2>(), f->item_count.as<int>());
  LPM_HIP(ctx, hipGetLastError());
  return LPM_OK;
}

// velocity of the current/stage state by `mode`: 0 plain, 1 expansion, 2 expansion + MLP
int ff_eval(lpm_bve_ff* f, int mode, const double* x, const double* y, const double* z, const double* q, double* u,
            double* v, double* w) {
  lpm_ctx* ctx = f->ctx;
  if (mode == 0) {
    lpm::PairProblem pp;
    pp.kind = LPM_K_SPHERE_BS;
    pp.precision = LPM_PREC_FP32_KAHAN;
    pp.n = f->n;
    pp.i0 = 0;
    pp.i1 = f->n;
    pp.x = x;
    pp.y = y;
    pp.z = z;
    pp.q0 = q;
    pp.area = f->area.as<double>();
    pp.src_list = f->list_plain.as<int>();
    pp.ns = f->ns;
    pp.radius = f->radius;
    pp.on_sphere = true;
    pp.out0 = u;
    pp.out1 = v;
    pp.out2 = w;
    pp.tgt_buf = &f->tgt_plain;
    pp.src_buf = &f->src_plain;
    pp.partial_buf = &f->partial_plain;
    return lpm::run_pair_sum(ctx, pp);
  }
  const int nc = f->ncell;
  dim3 b256(256);
  if (int rc = ff_bin(f, x, y, z)) return rc;
  hipLaunchKernelGGL(ff_pack_targets, dim3((f->n + 255) / 256), b256, 0, ctx->stream, f->n, f->tgt_perm.as<int>(), x,
                     y, z, f->trec.as<lpm::Vec4<float>>());
  lpm::PackArgs pa{x, y, z, q, nullptr, f->area.as<double>(), nullptr, f->src_perm.as<int>(), 0, 0, f->radius, 1.0};
  lpm::launch_pack(LPM_K_SPHERE_BS, LPM_PREC_FP32_KAHAN, pa, f->srec.p, nullptr, f->ns, 0, ctx->stream);
  GeomArgs ga{nc, f->src_perm.as<int>(), f->src_start.as<int>(), f->tgt_perm.as<int>(), f->tgt_start.as<int>(),
              x, y, z, q, f->area.as<double>(), f->radius, f->far_rec.as<float>(), f->mlp_rec.as<float>(),
              f->adir.as<double>(), f->geo.as<double>(), f->cen64.as<double>(), f->mom64.as<double>(),
              f->pgeo.as<double>()};
  hipLaunchKernelGGL(ff_cell_geometry, dim3(nc + f->npar), b256, 0, ctx->stream, ga);
  ClassArgs ca{nc, f->geo.as<double>(), f->r_near, f->r_band, f->near_list.as<int>(),
               f->near_count.as<int>(), f->band_list.as<int>(), f->band_count.as<int>()};
  hipLaunchKernelGGL(ff_classify, dim3(nc), b256, 0, ctx->stream, ca);
  FarListArgs la{nc, f->npar ? 4 : 1, f->geo.as<double>(), f->pgeo.as<double>(), f->r_near, f->r_band, f->r_par,
                 f->far_list.as<int>(), f->far_count.as<int>()};
  hipLaunchKernelGGL(ff_far_list, dim3(nc), b256, 0, ctx->stream, la);
  NearArgs na{f->trec.as<lpm::Vec4<float>>(), f->tgt_perm.as<int>(), f->tgt_start.as<int>(), f->srec.as<float>(),
              f->src_start.as<int>(), f->near_list.as<int>(), f->near_count.as<int>(), f->items.as<int2>(),
              f->item_count.as<int>(), nc, f->Vpart.as<double>(), f->n, f->near_split};
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (ctx->timing) {
    e0 = lpm::take_event(ctx);
    e1 = lpm::take_event(ctx);
    if (e0 && e1) LPM_HIP(ctx, hipEventRecord(e0, ctx->stream));
  }
  hipLaunchKernelGGL(ff_near_kernel, dim3((f->n_items + 3) / 4, f->near_split), b256, 0, ctx->stream, na);
  FarArgs fa{f->trec.as<lpm::Vec4<float>>(), f->tgt_start.as<int>(), f->far_rec.as<float>(), f->far_list.as<int>(),
             f->far_count.as<int>(), f->items.as<int2>(), f->item_count.as<int>(), nc, f->n,
             f->Vpart.as<double>() + (size_t)f->near_split * 3 * f->n};
  const dim3 gfar((f->n_items + 3) / 4, f->far_split);
  if (f->order == 2) hipLaunchKernelGGL(ff_far_kernel<2>, gfar, b256, 0, ctx->stream, fa);
  else if (f->order == 3) hipLaunchKernelGGL(ff_far_kernel<3>, gfar, b256, 0, ctx->stream, fa);
  else hipLaunchKernelGGL(ff_far_kernel<4>, gfar, b256, 0, ctx->stream, fa);
  int nparts = f->near_split + f->far_split;
  if (mode == 2 && f->trained) {
    MlpCorrArgs ma{f->trec.as<lpm::Vec4<float>>(), f->tgt_start.as<int>(), f->mlp_rec.as<float>(),
                   f->band_list.as<int>(), f->band_count.as<int>(), f->mlp_items.as<int2>(), f->item_count.as<int>() + 1, nc, f->n,
                   f->order,
                   f->net.frag.as<lpm::mlp_t>(), f->net.bias.as<float>(), f->Vpart.as<double>() + (size_t)3 * nparts * f->n};
    ++nparts;
    hipLaunchKernelGGL(ff_mlp_kernel, dim3(ctx->num_cus), dim3(512), 0, ctx->stream, ma);
  }
  if (ctx->timing && e0 && e1) {
    LPM_HIP(ctx, hipEventRecord(e1, ctx->stream));
    ctx->pending.push_back({e0, e1, LPM_K_FAR_FIELD});
  }
  hipLaunchKernelGGL(ff_epilogue, dim3((f->n + 255) / 256), b256, 0, ctx->stream, f->n, nparts, f->tgt_perm.as<int>(),
                     f->Vpart.as<double>(), x, y, z, u, v, w);
  LPM_HIP(ctx, hipGetLastError());
  return LPM_OK;
}

int ff_step(lpm_bve_ff* f, double dt, int mode) {
  lpm_ctx* ctx = f->ctx;
  const int n = f->n;
  dim3 g((n + 255) / 256), b(256);
  auto K = [&](int s, int c) { return f->k[s][c].as<double>(); };
  hipLaunchKernelGGL(ff_stage, g, b, 0, ctx->stream, n, dt, f->omega, f->radius, 0.5, 1, 1, f->x.as<double>(),
                     f->y.as<double>(), f->z.as<double>(), f->q.as<double>(), f->u.as<double>(), f->v.as<double>(),
                     f->w.as<double>(), K(0, 0), K(0, 1), K(0, 2), K(0, 3), f->xi.as<double>(), f->yi.as<double>(),
                     f->zi.as<double>(), f->qi.as<double>());
  for (int s = 1; s < 4; ++s) {
    if (int rc = ff_eval(f, mode, f->xi.as<double>(), f->yi.as<double>(), f->zi.as<double>(), f->qi.as<double>(),
                         K(s, 0), K(s, 1), K(s, 2)))
      return rc;
    hipLaunchKernelGGL(ff_stage, g, b, 0, ctx->stream, n, dt, f->omega, f->radius, s == 1 ? 0.5 : 1.0, 0, s < 3 ? 1 : 0,
                       f->x.as<double>(), f->y.as<double>(), f->z.as<double>(), f->q.as<double>(), nullptr, nullptr,
                       nullptr, K(s, 0), K(s, 1), K(s, 2), K(s, 3), f->xi.as<double>(), f->yi.as<double>(),
                       f->zi.as<double>(), f->qi.as<double>());
  }
  hipLaunchKernelGGL(ff_combine, g, b, 0, ctx->stream, n, f->radius, f->x.as<double>(), f->y.as<double>(),
                     f->z.as<double>(), f->q.as<double>(), (const double* const*)f->ptrs.p);
  LPM_HIP(ctx, hipGetLastError());
  return ff_eval(f, mode, f->x.as<double>(), f->y.as<double>(), f->z.as<double>(), f->q.as<double>(), f->u.as<double>(),
                 f->v.as<double>(), f->w.as<double>());
}

int ff_error(lpm_bve_ff* f, const double* au, const double* av, const double* aw, const double* bu, const double* bv,
             const double* bw, double* err) {
  lpm_ctx* ctx = f->ctx;
  const int nb = 256;
  LPM_HIP(ctx, f->err_part.ensure(2 * nb * sizeof(double)));
  hipLaunchKernelGGL(ff_err_partial, dim3(nb), dim3(256), 0, ctx->stream, f->n, au, av, aw, bu, bv, bw,
                     f->err_part.as<double>());
  std::vector<double> h(2 * nb);
  LPM_HIP(ctx, hipMemcpyAsync(h.data(), f->err_part.p, h.size() * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  double d = 0.0, m = 0.0;
  for (int i = 0; i < nb; ++i) {
    d = std::max(d, h[2 * i]);
    m = std::max(m, h[2 * i + 1]);
  }
  *err = m > 0 ? d / m : d;
  return LPM_OK;
}

// Load a particle set (at creation, and after a remesh): everything sized by
// the particle count -- active list, work-item bounds, near-list splits, the
// radix-sort workspace and the particle arrays (grown, never shrunk) -- then
// the plain velocity of the set (as BVESolver New) and its binning.  The
// cells, their frames, the network and the collected samples are kept.
int ff_load(lpm_bve_ff* f, int n, const double* x, const double* y, const double* z, const double* relvort,
            const double* area, const int32_t* active) {
  lpm_ctx* ctx = f->ctx;
  const int ncell = f->ncell;
  f->loaded = false;
  f->n = n;
  std::vector<int> plain;
  std::vector<int32_t> act((size_t)n);
  for (int i = 0; i < n; ++i) {
    act[(size_t)i] = active[i] ? 1 : 0;
    if (active[i]) plain.push_back(i);
  }
  f->ns = (int)plain.size();
  // work-item upper bounds: per cell ceil(count / tile) <= count / tile + 1
  f->n_items = ncell + n / (64 * kR) + 1;
  f->n_mlp_items = ncell + n / kMlpTile + 1;
  // near-list and far-cell splits: about kSplitRounds rounds of each kernel's
  // resident waves
  {
    const double waves = (double)n / (64 * kR) + 0.5 * ncell;
    auto split_for = [&](const void* kernel) {
      int nb = 0;
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, 256, 0) != hipSuccess || nb <= 0) nb = 1;
      const double slots = (double)nb * 4 * ctx->num_cus;
      return std::min(kSplitMax, std::max(1, (int)std::ceil(kSplitRounds * slots / std::max(waves, 1.0))));
    };
    f->near_split = split_for(reinterpret_cast<const void*>(ff_near_kernel));
    f->far_split = split_for(f->order == 2   ? reinterpret_cast<const void*>(ff_far_kernel<2>)
                             : f->order == 3 ? reinterpret_cast<const void*>(ff_far_kernel<3>)
                                             : reinterpret_cast<const void*>(ff_far_kernel<4>));
  }
  const size_t nb = (size_t)n * sizeof(double);
  const size_t ni = (size_t)n * sizeof(int);
  int rc = LPM_OK;
  auto chk = [&](int r) {
    if (r && !rc) rc = r;
    return rc == LPM_OK;
  };
  chk(ff_upload(ctx, f->x, x, nb)) && chk(ff_upload(ctx, f->y, y, nb)) && chk(ff_upload(ctx, f->z, z, nb)) &&
      chk(ff_upload(ctx, f->q, relvort, nb)) && chk(ff_upload(ctx, f->area, area, nb)) &&
      chk(ff_upload(ctx, f->u, nullptr, nb)) && chk(ff_upload(ctx, f->v, nullptr, nb)) &&
      chk(ff_upload(ctx, f->w, nullptr, nb)) && chk(ff_upload(ctx, f->pu, nullptr, nb)) &&
      chk(ff_upload(ctx, f->pv, nullptr, nb)) && chk(ff_upload(ctx, f->pw, nullptr, nb)) &&
      chk(ff_upload(ctx, f->xi, nullptr, nb)) && chk(ff_upload(ctx, f->yi, nullptr, nb)) &&
      chk(ff_upload(ctx, f->zi, nullptr, nb)) && chk(ff_upload(ctx, f->qi, nullptr, nb)) &&
      chk(ff_upload(ctx, f->src_perm, nullptr, ni)) &&
      chk(ff_upload(ctx, f->src_start, nullptr, ((size_t)ncell + 1) * 4)) &&
      chk(ff_upload(ctx, f->tgt_perm, nullptr, ni)) &&
      chk(ff_upload(ctx, f->tgt_start, nullptr, ((size_t)ncell + 1) * 4)) &&
      chk(ff_upload(ctx, f->cellof, nullptr, ni)) &&
      chk(ff_upload(ctx, f->active, act.data(), ni)) &&
      chk(ff_upload(ctx, f->sort_tmp, nullptr, lpm::cell_sort_bytes(n))) &&
      chk(ff_upload(ctx, f->item_count, nullptr, 2 * 4)) &&
      chk(ff_upload(ctx, f->list_plain, plain.data(), std::max<size_t>(plain.size(), 1) * 4)) &&
      chk(ff_upload(ctx, f->items, nullptr, (size_t)f->n_items * sizeof(int2))) &&
      chk(ff_upload(ctx, f->mlp_items, nullptr, (size_t)f->n_mlp_items * sizeof(int2))) &&
      chk(ff_upload(ctx, f->trec, nullptr, (size_t)n * 16)) &&
      chk(ff_upload(ctx, f->srec, nullptr, std::max<size_t>((size_t)f->ns, 1) * lpm::SREC * 4)) &&
      chk(ff_upload(ctx, f->far_rec, nullptr, (size_t)(ncell + ncell / 4) * kCellRec * 4)) &&
      chk(ff_upload(ctx, f->mlp_rec, nullptr, (size_t)ncell * kMlpRec * 4)) &&
      chk(ff_upload(ctx, f->geo, nullptr, (size_t)ncell * 8 * 8)) &&
      chk(ff_upload(ctx, f->cen64, nullptr, (size_t)ncell * 3 * 8)) &&
      chk(ff_upload(ctx, f->mom64, nullptr, (size_t)ncell * kNMom * 8)) &&
      chk(ff_upload(ctx, f->far_list, nullptr, (size_t)ncell * ncell * 4)) &&
      chk(ff_upload(ctx, f->far_count, nullptr, (size_t)ncell * 4)) &&
      chk(ff_upload(ctx, f->near_list, nullptr, (size_t)ncell * ncell * 4)) &&
      chk(ff_upload(ctx, f->near_count, nullptr, (size_t)ncell * 4)) &&
      chk(ff_upload(ctx, f->band_list, nullptr, (size_t)ncell * ncell * 4)) &&
      chk(ff_upload(ctx, f->band_count, nullptr, (size_t)ncell * 4)) &&
      chk(ff_upload(ctx, f->Vpart, nullptr, (size_t)(f->near_split + f->far_split + 1) * 3 * nb));
  for (int s = 0; s < 4 && rc == LPM_OK; ++s)
    for (int c = 0; c < 4 && rc == LPM_OK; ++c) chk(ff_upload(ctx, f->k[s][c], nullptr, nb));
  if (rc == LPM_OK) {
    std::vector<double*> tab(16);
    for (int c = 0; c < 4; ++c)
      for (int s = 0; s < 4; ++s) tab[(size_t)(c * 4 + s)] = f->k[s][c].as<double>();
    chk(ff_upload(ctx, f->ptrs, tab.data(), tab.size() * sizeof(double*)));
    hipError_t e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) rc = lpm::hip_fail(ctx, e, "hipStreamSynchronize");
  }
  if (rc == LPM_OK) {
    // start on the sphere, with the plain velocity stored (as BVESolver New)
    hipLaunchKernelGGL(ff_project, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, n, f->radius,
                       f->x.as<double>(), f->y.as<double>(), f->z.as<double>());
    chk(ff_eval(f, 0, f->x.as<double>(), f->y.as<double>(), f->z.as<double>(), f->q.as<double>(), f->u.as<double>(),
                f->v.as<double>(), f->w.as<double>()));
    // bin once so that the cell queries are defined before any evaluation
    if (rc == LPM_OK) chk(ff_bin(f, f->x.as<double>(), f->y.as<double>(), f->z.as<double>()));
  }
  if (rc == LPM_OK) {
    hipError_t e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) rc = lpm::hip_fail(ctx, e, "hipStreamSynchronize");
  }
  f->loaded = rc == LPM_OK;
  return rc;
}

int ff_usable(lpm_bve_ff* f) {
  if (f->loaded) return LPM_OK;
  return fail(f->ctx, LPM_ERR_STATE, "far-field particles were not loaded (a particle reload failed)");
}

}  // namespace

extern "C" {

int lpm_bve_ff_new(lpm_ctx* ctx, lpm_bve_ff** out, int n, const double* x, const double* y, const double* z,
                   const double* relvort, const double* area, const int32_t* active, const int32_t* cell, int ncell,
                   double radius, double rotation_rate, double near_radius, double band_radius, int flags) {
  if (!ctx || !out) return LPM_ERR_ARG;
  ctx->err.clear();
  *out = nullptr;
  if (n <= 0 || ncell <= 0 || !x || !y || !z || !relvort || !area || !active || !cell)
    return fail(ctx, LPM_ERR_ARG, "lpm_bve_ff_new: bad arguments");
  if (!(radius > 0.0) || !(near_radius >= 0.0) || !(band_radius >= near_radius))
    return fail(ctx, LPM_ERR_ARG, "lpm_bve_ff_new: need radius > 0 and 0 <= near_radius <= band_radius");
  const int order = (flags & LPM_FF_ORDER_MASK) == 0 ? 4 : (flags & LPM_FF_ORDER_MASK);
  if (order < 2 || order > 4 || (flags & ~(LPM_FF_ORDER_MASK | LPM_FF_SAMPLE_DRAWS_MASK)))
    return fail(ctx, LPM_ERR_ARG,
                "lpm_bve_ff_new: flags hold the expansion order 2, 3 or 4 (0: 4) and the sample draws only");
  const int draws = std::max(1, (flags & LPM_FF_SAMPLE_DRAWS_MASK) >> 3);
  for (int i = 0; i < n; ++i)
    if (cell[i] < 0 || cell[i] >= ncell) return fail(ctx, LPM_ERR_ARG, "lpm_bve_ff_new: cell id out of range");
  LPM_HIP(ctx, hipSetDevice(ctx->device));
  lpm_bve_ff* f = new lpm_bve_ff();
  f->ctx = ctx;
  f->n = n;
  f->ncell = ncell;
  f->radius = radius;
  f->omega = rotation_rate;
  f->r_near = near_radius;
  f->r_band = band_radius;
  f->order = order;
  f->draws = draws;
  // Cells are fixed regions of the sphere: each is the set of points nearest to
  // its generator, the direction of the area-weighted centroid of the given
  // cell's active sources at set-up (of all its particles if it has none).  Its
  // frame anchor is the direction of its active source farthest from that
  // centroid (lowest particle index on ties).  Particles are binned anew at
  // every evaluation, so cells never stretch with the flow.
  std::vector<lpm::Vec4<float>> gen((size_t)ncell);
  std::vector<double> adir((size_t)ncell * 3, 0.0);
  {
    std::vector<double> cs((size_t)ncell * 4, 0.0), ca((size_t)ncell * 4, 0.0);
    for (int i = 0; i < n; ++i) {
      double* c = &ca[(size_t)cell[i] * 4];
      c[0] += x[i];
      c[1] += y[i];
      c[2] += z[i];
      c[3] += 1.0;
      if (active[i]) {
        double* s = &cs[(size_t)cell[i] * 4];
        s[0] += area[i] * x[i];
        s[1] += area[i] * y[i];
        s[2] += area[i] * z[i];
        s[3] += area[i];
      }
    }
    std::vector<double> best((size_t)ncell, -1.0);
    for (int i = 0; i < n; ++i)
      if (active[i]) {
        const double* c = &cs[(size_t)cell[i] * 4];
        const double inv = c[3] > 0 ? 1.0 / c[3] : 0.0;
        const double dx = x[i] - c[0] * inv, dy = y[i] - c[1] * inv, dz = z[i] - c[2] * inv;
        const double d2 = dx * dx + dy * dy + dz * dz;
        if (d2 > best[(size_t)cell[i]]) {
          best[(size_t)cell[i]] = d2;
          const double r = std::sqrt(x[i] * x[i] + y[i] * y[i] + z[i] * z[i]);
          adir[(size_t)cell[i] * 3 + 0] = x[i] / r;
          adir[(size_t)cell[i] * 3 + 1] = y[i] / r;
          adir[(size_t)cell[i] * 3 + 2] = z[i] / r;
        }
      }
    for (int c = 0; c < ncell; ++c) {
      const double* s = cs[(size_t)c * 4 + 3] > 0 ? &cs[(size_t)c * 4] : &ca[(size_t)c * 4];
      const double r = std::sqrt(s[0] * s[0] + s[1] * s[1] + s[2] * s[2]);
      if (r > 0) gen[(size_t)c] = lpm::Vec4<float>{(float)(s[0] / r), (float)(s[1] / r), (float)(s[2] / r), 0.f};
      else gen[(size_t)c] = lpm::Vec4<float>{0.f, 0.f, 0.f, 0.f};  // empty cell: never nearest
    }
  }
  int rc = LPM_OK;
  auto chk = [&](int r) {
    if (r && !rc) rc = r;
    return rc == LPM_OK;
  };
  const int g = loc_grid(ncell), nbins = 6 * g * g;
  if (chk(ff_upload(ctx, f->gen, gen.data(), (size_t)ncell * sizeof(lpm::Vec4<float>))) &&
      chk(ff_upload(ctx, f->bins, nullptr, (size_t)nbins * sizeof(LocBin)))) {
    hipLaunchKernelGGL(ff_locate_bins, dim3((nbins + 255) / 256), dim3(256), 0, ctx->stream, ncell, g,
                       f->gen.as<lpm::Vec4<float>>(), f->bins.as<LocBin>());
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) rc = lpm::hip_fail(ctx, e, "ff_locate_bins");
  }
  chk(rc) && chk(ff_upload(ctx, f->adir, adir.data(), adir.size() * 8)) && chk(f->net.init(ctx, 13, 128, 3, 3, LPM_ACT_ISRU, 12345)) &&
      chk(ff_load(f, n, x, y, z, relvort, area, active));
  if (rc != LPM_OK) {
    lpm_bve_ff_delete(f);
    return rc;
  }
  *out = f;
  return lpm::collect_timing(ctx);
}

int lpm_bve_ff_velocity(lpm_bve_ff* f, int mode, double* u, double* v, double* w) {
  if (!f || !u || !v || !w) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  ctx->err.clear();
  if (int rc = ff_usable(f)) return rc;
  if (mode < 0 || mode > 2) return fail(ctx, LPM_ERR_ARG, "lpm_bve_ff_velocity: mode must be 0, 1 or 2");
  if (mode == 2 && !f->trained) return fail(ctx, LPM_ERR_STATE, "lpm_bve_ff_velocity: the network is not trained");
  LPM_HIP(ctx, hipSetDevice(ctx->device));
  if (int rc = ff_eval(f, mode, f->x.as<double>(), f->y.as<double>(), f->z.as<double>(), f->q.as<double>(),
                       f->pu.as<double>(), f->pv.as<double>(), f->pw.as<double>()))
    return rc;
  const size_t nb = (size_t)f->n * sizeof(double);
  LPM_HIP(ctx, hipMemcpyAsync(u, f->pu.p, nb, hipMemcpyDeviceToHost, ctx->stream));
  LPM_HIP(ctx, hipMemcpyAsync(v, f->pv.p, nb, hipMemcpyDeviceToHost, ctx->stream));
  LPM_HIP(ctx, hipMemcpyAsync(w, f->pw.p, nb, hipMemcpyDeviceToHost, ctx->stream));
  LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return lpm::collect_timing(ctx);
}

int lpm_bve_ff_collect(lpm_bve_ff* f, int n_samples, uint64_t seed, int64_t* total) {
  if (!f || n_samples <= 0) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  ctx->err.clear();
  if (int rc = ff_usable(f)) return rc;
  LPM_HIP(ctx, hipSetDevice(ctx->device));
  // refresh geometry, moments and lists at the current state (expansion mode)
  if (int rc = ff_eval(f, 1, f->x.as<double>(), f->y.as<double>(), f->z.as<double>(), f->q.as<double>(),
                       f->pu.as<double>(), f->pv.as<double>(), f->pw.as<double>()))
    return rc;
  const int64_t need = f->n_collected + n_samples;
  if (need > f->cap_collected) {
    const int64_t cap = std::max<int64_t>(need, 2 * f->cap_collected);
    DevBuf nx, ny, ni;
    LPM_HIP(ctx, nx.ensure((size_t)cap * 13 * 4));
    LPM_HIP(ctx, ny.ensure((size_t)cap * 3 * 4));
    LPM_HIP(ctx, ni.ensure((size_t)cap * 2 * 4));
    if (f->n_collected > 0) {
      LPM_HIP(ctx, hipMemcpyAsync(nx.p, f->sx.p, (size_t)f->n_collected * 13 * 4, hipMemcpyDeviceToDevice, ctx->stream));
      LPM_HIP(ctx, hipMemcpyAsync(ny.p, f->sy.p, (size_t)f->n_collected * 3 * 4, hipMemcpyDeviceToDevice, ctx->stream));
      LPM_HIP(ctx, hipMemcpyAsync(ni.p, f->sid.p, (size_t)f->n_collected * 2 * 4, hipMemcpyDeviceToDevice, ctx->stream));
    }
    LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    f->sx.release();
    f->sy.release();
    f->sid.release();
    f->sx = nx;
    f->sy = ny;
    f->sid = ni;
    nx.p = ny.p = ni.p = nullptr;
    f->cap_collected = cap;
  }
  SampleArgs sa{n_samples, (unsigned long long)seed, f->n, f->ncell, f->order, f->tgt_perm.as<int>(), f->tgt_cell,
                f->src_perm.as<int>(), f->src_start.as<int>(), f->band_list.as<int>(), f->band_count.as<int>(),
                f->x.as<double>(), f->y.as<double>(), f->z.as<double>(), f->q.as<double>(), f->area.as<double>(),
                f->cen64.as<double>(), f->mom64.as<double>(), f->mlp_rec.as<float>(), f->radius,
                f->sx.as<float>() + (size_t)f->n_collected * 13, f->sy.as<float>() + (size_t)f->n_collected * 3,
                f->sid.as<int>() + (size_t)f->n_collected * 2};
  sa.draws = f->draws;
  hipLaunchKernelGGL(ff_make_samples, dim3((n_samples + 255) / 256), dim3(256), 0, ctx->stream, sa);
  LPM_HIP(ctx, hipGetLastError());
  LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  f->n_collected += n_samples;
  if (total) *total = f->n_collected;
  return LPM_OK;
}

int lpm_bve_ff_train(lpm_bve_ff* f, int epochs, int batch, double lr, uint64_t seed, double* final_loss) {
  if (!f || epochs < 0 || batch <= 0) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  ctx->err.clear();
  if (f->n_collected <= 0) return fail(ctx, LPM_ERR_STATE, "lpm_bve_ff_train: no samples collected");
  if (f->n_collected > INT32_MAX) return fail(ctx, LPM_ERR_ARG, "lpm_bve_ff_train: too many samples");
  LPM_HIP(ctx, hipSetDevice(ctx->device));
  // targets are trained at unit RMS (scale fixed at the first training); the
  // stored parameters keep the scale folded into the output layer
  if (!(f->ys > 0.0)) {
    double r = 0.0;
    if (int rc = f->net.rms(f->n_collected * 3, f->sy.as<float>(), &r)) return rc;
    f->ys = r > 0.0 ? r : 1.0;
  }
  if (f->trained)
    if (int rc = f->net.scale_output((float)(1.0 / f->ys))) return rc;
  if (int rc = f->net.train((int)f->n_collected, f->sx.as<float>(), f->sy.as<float>(), epochs, batch, (float)lr, seed,
                            final_loss, nullptr, true, (float)(1.0 / f->ys)))
    return rc;
  if (int rc = f->net.scale_output((float)f->ys)) return rc;
  if (int rc = f->net.pack()) return rc;
  LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  f->trained = true;
  return LPM_OK;
}

int lpm_bve_ff_set_online(lpm_bve_ff* f, int n_samples, int epochs, int batch, double lr) {
  if (!f || n_samples < 0 || epochs < 0 || batch <= 0 || !(lr >= 0.0)) return LPM_ERR_ARG;
  f->online_n = n_samples;
  f->online_epochs = epochs;
  f->online_batch = batch;
  f->online_lr = lr;
  return LPM_OK;
}

int lpm_bve_ff_set_online_from(lpm_bve_ff* f, double fraction) {
  if (!f || !(fraction >= 0.0 && fraction <= 1.0)) return LPM_ERR_ARG;
  f->online_from = fraction;
  return LPM_OK;
}

int lpm_bve_ff_set_params(lpm_bve_ff* f, const float* params, int64_t count) {
  if (!f || !params) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  if (count != f->net.np) return fail(ctx, LPM_ERR_ARG, "lpm_bve_ff_set_params: wrong parameter count");
  LPM_HIP(ctx, hipMemcpyAsync(f->net.p.p, params, (size_t)count * 4, hipMemcpyHostToDevice, ctx->stream));
  if (int rc = f->net.pack()) return rc;
  LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  f->trained = true;
  return LPM_OK;
}

int lpm_bve_ff_get_params(lpm_bve_ff* f, float* params, int64_t count) {
  if (!f || !params) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  if (count != f->net.np) return fail(ctx, LPM_ERR_ARG, "lpm_bve_ff_get_params: wrong parameter count");
  LPM_HIP(ctx, hipMemcpyAsync(params, f->net.p.p, (size_t)count * 4, hipMemcpyDeviceToHost, ctx->stream));
  LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return LPM_OK;
}

int lpm_bve_ff_samples(lpm_bve_ff* f, int64_t offset, int64_t count, float* in, float* target, int32_t* ids) {
  if (!f || !in || !target || offset < 0 || count < 0 || offset + count > f->n_collected) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  LPM_HIP(ctx, hipMemcpyAsync(in, f->sx.as<float>() + (size_t)offset * 13, (size_t)count * 13 * 4,
                              hipMemcpyDeviceToHost, ctx->stream));
  LPM_HIP(ctx, hipMemcpyAsync(target, f->sy.as<float>() + (size_t)offset * 3, (size_t)count * 3 * 4,
                              hipMemcpyDeviceToHost, ctx->stream));
  if (ids)
    LPM_HIP(ctx, hipMemcpyAsync(ids, f->sid.as<int>() + (size_t)offset * 2, (size_t)count * 2 * 4,
                                hipMemcpyDeviceToHost, ctx->stream));
  LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return LPM_OK;
}

int lpm_bve_ff_steps(lpm_bve_ff* f, double dt, int nsteps, int mode, int judge_every, double tol, int* mode_out,
                     double* last_error, int* judged) {
  if (!f || nsteps < 0) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  ctx->err.clear();
  if (int rc = ff_usable(f)) return rc;
  if (mode < 0 || mode > 2) return fail(ctx, LPM_ERR_ARG, "lpm_bve_ff_steps: mode must be 0, 1 or 2");
  if (mode == 2 && !f->trained) return fail(ctx, LPM_ERR_STATE, "lpm_bve_ff_steps: the network is not trained");
  LPM_HIP(ctx, hipSetDevice(ctx->device));
  int cur = mode, nj = 0;
  double err = -1.0;
  for (int s = 1; s <= nsteps; ++s) {
    if (int rc = ff_step(f, dt, cur)) return rc;
    if (cur != 0 && judge_every > 0 && s % judge_every == 0) {
      // the plain direct sum judges the stored velocity; above tol fall back for good
      if (int rc = ff_eval(f, 0, f->x.as<double>(), f->y.as<double>(), f->z.as<double>(), f->q.as<double>(),
                           f->pu.as<double>(), f->pv.as<double>(), f->pw.as<double>()))
        return rc;
      if (int rc = ff_error(f, f->u.as<double>(), f->v.as<double>(), f->w.as<double>(), f->pu.as<double>(),
                            f->pv.as<double>(), f->pw.as<double>(), &err))
        return rc;
      ++nj;
      if (!(err <= tol)) {
        cur = 0;
        LPM_HIP(ctx, hipMemcpyAsync(f->u.p, f->pu.p, (size_t)f->n * 8, hipMemcpyDeviceToDevice, ctx->stream));
        LPM_HIP(ctx, hipMemcpyAsync(f->v.p, f->pv.p, (size_t)f->n * 8, hipMemcpyDeviceToDevice, ctx->stream));
        LPM_HIP(ctx, hipMemcpyAsync(f->w.p, f->pw.p, (size_t)f->n * 8, hipMemcpyDeviceToDevice, ctx->stream));
      } else if (cur == 2 && f->online_n > 0 && err > f->online_from * tol) {
        // fine-tune on direct sums of the judged state for the steps that follow
        f->n_collected = 0;
        if (int rc = lpm_bve_ff_collect(f, f->online_n, 0x5eedull + (uint64_t)(++f->online_rounds), nullptr))
          return rc;
        if (f->online_epochs > 0)
          if (int rc = lpm_bve_ff_train(f, f->online_epochs, f->online_batch, f->online_lr,
                                        (uint64_t)f->online_rounds, nullptr))
            return rc;
      }
    }
  }
  LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (mode_out) *mode_out = cur;
  if (last_error) *last_error = err;
  if (judged) *judged = nj;
  return lpm::collect_timing(ctx);
}

int lpm_bve_ff_get_state(lpm_bve_ff* f, double* x, double* y, double* z, double* relvort, double* u, double* v,
                         double* w) {
  if (!f) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  ctx->err.clear();
  if (int rc = ff_usable(f)) return rc;
  const DevBuf* src[7] = {&f->x, &f->y, &f->z, &f->q, &f->u, &f->v, &f->w};
  double* dst[7] = {x, y, z, relvort, u, v, w};
  for (int k = 0; k < 7; ++k)
    if (dst[k])
      LPM_HIP(ctx, hipMemcpyAsync(dst[k], src[k]->p, (size_t)f->n * 8, hipMemcpyDeviceToHost, ctx->stream));
  LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return LPM_OK;
}

int lpm_bve_ff_set_particles(lpm_bve_ff* f, int n, const double* x, const double* y, const double* z,
                             const double* relvort, const double* area, const int32_t* active) {
  if (!f) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  ctx->err.clear();
  if (n <= 0 || !x || !y || !z || !relvort || !area || !active)
    return fail(ctx, LPM_ERR_ARG, "lpm_bve_ff_set_particles: n must be > 0 and the arrays non-null");
  LPM_HIP(ctx, hipSetDevice(ctx->device));
  if (int rc = ff_load(f, n, x, y, z, relvort, area, active)) return rc;
  return lpm::collect_timing(ctx);
}

int lpm_bve_ff_set_state(lpm_bve_ff* f, const double* x, const double* y, const double* z, const double* relvort) {
  if (!f || !x || !y || !z || !relvort) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  ctx->err.clear();
  if (int rc = ff_usable(f)) return rc;
  LPM_HIP(ctx, hipSetDevice(ctx->device));
  const size_t nb = (size_t)f->n * sizeof(double);
  LPM_HIP(ctx, hipMemcpyAsync(f->x.p, x, nb, hipMemcpyHostToDevice, ctx->stream));
  LPM_HIP(ctx, hipMemcpyAsync(f->y.p, y, nb, hipMemcpyHostToDevice, ctx->stream));
  LPM_HIP(ctx, hipMemcpyAsync(f->z.p, z, nb, hipMemcpyHostToDevice, ctx->stream));
  LPM_HIP(ctx, hipMemcpyAsync(f->q.p, relvort, nb, hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(ff_project, dim3((f->n + 255) / 256), dim3(256), 0, ctx->stream, f->n, f->radius,
                     f->x.as<double>(), f->y.as<double>(), f->z.as<double>());
  if (int rc = ff_eval(f, 0, f->x.as<double>(), f->y.as<double>(), f->z.as<double>(), f->q.as<double>(),
                       f->u.as<double>(), f->v.as<double>(), f->w.as<double>()))
    return rc;
  LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return lpm::collect_timing(ctx);
}

int lpm_bve_ff_particle_cells(lpm_bve_ff* f, int32_t* cell) {
  if (!f || !cell) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  ctx->err.clear();
  if (int rc = ff_usable(f)) return rc;
  LPM_HIP(ctx, hipSetDevice(ctx->device));
  LPM_HIP(ctx, hipMemcpyAsync(cell, f->cellof.p, (size_t)f->n * 4, hipMemcpyDeviceToHost, ctx->stream));
  LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return LPM_OK;
}

int lpm_bve_ff_cells(lpm_bve_ff* f, int* near_cells, int* band_cells) {
  if (!f || !near_cells || !band_cells) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  ctx->err.clear();
  if (int rc = ff_usable(f)) return rc;
  LPM_HIP(ctx, hipSetDevice(ctx->device));
  LPM_HIP(ctx, hipMemcpyAsync(near_cells, f->near_count.p, (size_t)f->ncell * 4, hipMemcpyDeviceToHost, ctx->stream));
  LPM_HIP(ctx, hipMemcpyAsync(band_cells, f->band_count.p, (size_t)f->ncell * 4, hipMemcpyDeviceToHost, ctx->stream));
  LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return LPM_OK;
}

int lpm_bve_ff_set_parents(lpm_bve_ff* f, double parent_radius) {
  if (!f) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  ctx->err.clear();
  if (!(parent_radius >= 0.0)) return fail(ctx, LPM_ERR_ARG, "lpm_bve_ff_set_parents: parent_radius must be >= 0");
  if (parent_radius > 0.0 && f->ncell % 4 != 0)
    return fail(ctx, LPM_ERR_ARG, "lpm_bve_ff_set_parents: the coarse level needs a cell count divisible by 4");
  LPM_HIP(ctx, hipSetDevice(ctx->device));
  if (parent_radius > 0.0) LPM_HIP(ctx, f->pgeo.ensure((size_t)(f->ncell / 4) * 4 * sizeof(double)));
  f->r_par = parent_radius;
  f->npar = parent_radius > 0.0 ? f->ncell / 4 : 0;
  return LPM_OK;
}

int lpm_bve_ff_far_counts(lpm_bve_ff* f, int* far_records) {
  if (!f || !far_records) return LPM_ERR_ARG;
  lpm_ctx* ctx = f->ctx;
  ctx->err.clear();
  if (int rc = ff_usable(f)) return rc;
  LPM_HIP(ctx, hipSetDevice(ctx->device));
  LPM_HIP(ctx, hipMemcpyAsync(far_records, f->far_count.p, (size_t)f->ncell * 4, hipMemcpyDeviceToHost, ctx->stream));
  LPM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return LPM_OK;
}

int lpm_bve_ff_delete(lpm_bve_ff* f) {
  if (!f) return LPM_ERR_ARG;
  (void)hipStreamSynchronize(f->ctx->stream);
  DevBuf* all[] = {&f->x, &f->y, &f->z, &f->q, &f->u, &f->v, &f->w, &f->area, &f->xi, &f->yi, &f->zi, &f->qi,
                   &f->pu, &f->pv, &f->pw, &f->src_perm, &f->src_start, &f->tgt_perm, &f->tgt_start,
                   &f->trec, &f->srec, &f->far_rec, &f->mlp_rec, &f->geo, &f->cen64, &f->mom64, &f->far_list, &f->far_count, &f->pgeo,
                   &f->near_list, &f->near_count, &f->band_list, &f->band_count, &f->items, &f->mlp_items,
                   &f->list_plain, &f->tgt_plain, &f->src_plain, &f->partial_plain, &f->ptrs, &f->err_part, &f->sx,
                   &f->sy, &f->sid, &f->cellof, &f->active,
                   &f->sort_tmp, &f->item_count, &f->gen, &f->bins, &f->adir, &f->Vpart};
  for (DevBuf* b : all) b->release();
  for (auto& row : f->k)
    for (auto& b : row) b.release();
  delete f;
  return LPM_OK;
}

}  // extern "C"
