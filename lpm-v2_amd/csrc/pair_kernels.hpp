// pair_kernels.hpp -- tiled all-pairs direct-sum kernels for gfx950.
//
// One template covers every O(T*S) sum of the path.  A "pair policy" P
// supplies the per-pair arithmetic; the template supplies the CDNA4 mapping:
//
//  * a wavefront owns 64*R consecutive targets: lane l holds targets
//    t0 + r*64 + l (r < R) in registers, so each source value loaded is used
//    by 64*R pairs;
//  * sources are packed AoS records (8 words) read with wave-uniform
//    addresses, which the compiler turns into scalar (SMEM) loads: the source
//    operands of the pair arithmetic come straight from SGPRs and cost no
//    LDS or VGPR traffic;
//  * sources are walked in tiles of KT; inside a tile each target
//    accumulates plainly in FP32, and the tile partial is folded into a
//    (sum, compensation) pair with an error-free TwoSum (Knuth), so the
//    compensated accumulation costs O(S/KT) per target;
//  * the self pair j == i is excluded by index, exactly, but only tiles whose
//    source-index range overlaps the wave's target range take the checked
//    path (a wave-uniform branch);
//  * a grid of (target tiles) x (source splits) fills the 256 CUs also when T
//    is small; every split writes its FP64 partial per target and a
//    finalize kernel reduces the splits in a fixed order (deterministic).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lpm {

// Source records: P::NW words per source (FP32) or doubles (FP64); 8 unless
// a policy needs more.
//   sphere BS   : x y z e w2 idx . .     e = R^2-|x|^2, w2 = -zeta A/(2 pi R)
//   plane  BS   : x y w idx . . . .      w = omega A / (2 pi)
//   PSE         : x y fA A idx . . .     coordinates scaled (see PsePolicy)
//   sphere green: x y z e gr ga idx .    g = -zeta A ln2/(4 pi) (FP32) or -zeta A/(4 pi) (FP64)
//   plane  green: x y g idx . . . .      g = omega A ln2/(4 pi) (FP32) or omega A/(4 pi) (FP64)
//   PSE derivative, interpolation, SWE: see PseDeriv, PseInterp, SwePlane
// Target records: 4 words per target: sphere {x y z e}, plane {x y . .},
// PSE {x y f .}.
constexpr int SREC = 8;
constexpr int TREC = 4;
constexpr int SREC_MAX = 12;

template <typename T>
struct Vec4 {
  T a, b, c, d;
};

__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
// FP64 reciprocal: the hardware estimate r (v_rcp_f64, 2^-24.4) with the error
// e = 1 - x r taken out to third order, r (1 + e + e^2): what is left is e^3, 2^-73, so
// the result is within an ulp of the correctly rounded 1 / x for normal x.  Four
// instructions, against five for two Newton steps and about ten for the IEEE division
// sequence; x = 0 gives NaN instead of inf, which the pair sums multiply by a zero
// separation either way.
__device__ __forceinline__ double rcp_refined(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, r, 1.0);
  return fma(r, fma(e, e, e), r);
}
// Four reciprocals for the price of one: r = 1 / (z0 z1 z2 z3) and nine products, 72
// cycles against 120 for four refined ones.  Each is off by 0.66 ulp rms (at most 3)
// instead of 0.29, which stays below the roundings of the separations and the sums: rms
// errors against 80-bit sums at icosahedral L3 / L4 / L5 / L6 and the 300^2 plane are 2.01,
// 2.50, 4.89, 8.29 and 0.11e-15, before, one by one by two Newton steps, 2.01, 2.50, 4.89,
// 8.29 and 0.41e-15.  Where the product leaves the range of FP64 (coincident points, separations
// beyond 1e38 or below 1e-38) all four are NaN, and pair_tile takes the wave's sums
// again one by one.
__device__ __forceinline__ void rcp_four(const double z[4], double f[4]) {
  const double a = z[0] * z[1], b = z[2] * z[3], p = a * b;
  const double r = rcp_refined(p);
  const double ra = r * b, rb = r * a;
  f[0] = ra * z[1];
  f[1] = ra * z[0];
  f[2] = rb * z[3];
  f[3] = rb * z[2];
}
// FP64 exponential and logarithm by table.  The FP64 vector rate is 4.6 cycles per
// instruction and SIMD, so the sums below are bound by the length of these: a table
// entry from LDS (512 or 2,048 bytes, filled once per block) takes the place of half
// of the polynomial.  All pairs at icosahedral L6: Green sum 11.8 -> 8.1 ms; PSE-8 at
// 256^2: 3.6 -> 3.0 ms.  Kernels whose policy names a TABLE call fill_tables first.
enum Table { kNoTable = 0, kExpTable = 1, kLogTable = 2 };
constexpr int kExpBits = 6;  // 2^(i / 64)
constexpr int kLogBits = 7;  // {c_i, -log c_i}, c_i near 1 / m in the i-th 128th of [0.70, 1.41)

__device__ __forceinline__ double* exp_table() {
  __shared__ double t[1 << kExpBits];
  return t;
}
struct LogEntry {
  double c, l;
};
__device__ __forceinline__ LogEntry* log_table() {
  __shared__ LogEntry t[1 << kLogBits];
  return t;
}

// High word of the lower end of the mantissa interval, about sqrt(1/2).
constexpr unsigned kLogLow = 0x3fe66000u;

template <int TABLE>
__device__ __forceinline__ void fill_tables() {
  if constexpr (TABLE == kExpTable) {
    if (threadIdx.x < (1 << kExpBits)) exp_table()[threadIdx.x] = exp2(threadIdx.x / (double)(1 << kExpBits));
    __syncthreads();
  } else if constexpr (TABLE == kLogTable) {
    if (threadIdx.x < (1 << kLogBits)) {
      // the interval's middle; c has 9 bits so that c is exact in the product below,
      // and is 1 next to m = 1, where log m = log1p(m - 1) must not lose its own digits
      const unsigned step = 1u << (20 - kLogBits);
      const unsigned lo = kLogLow + threadIdx.x * step;
      const double m = __hiloint2double((int)(lo + step / 2), 0);
      const double m0 = __hiloint2double((int)lo, 0), m1 = __hiloint2double((int)(lo + step), 0);
      double c = rint(512.0 / m) / 512.0;
      if (m0 <= 1.0 && 1.0 <= m1) c = 1.0;
      log_table()[threadIdx.x] = LogEntry{c, c == 1.0 ? 0.0 : -log(c)};
    }
    __syncthreads();
  }
}

// exp(-q) for q >= 0: -q = (64 e + i) ln 2 / 64 + r, |r| <= ln 2 / 128, and
// exp r = 1 + r + ... + r^6 / 720 (first dropped term 2e-19); within an ulp of the
// correctly rounded value, 0 from q = 745.2 as the library's.  12 FP64 and 4 integer
// instructions against about 26.  NaN gives exp(-800) = 0 unless NAN_SAFE: the
// polynomial factor of the 8th-order kernels carries it.
template <bool NAN_SAFE = false>
__device__ __forceinline__ double exp_neg_fp64(double q) {
  constexpr double kInv = 92.332482616893656877;        // 64 / ln 2
  constexpr double kHi = 0.010830424696223417;          // ln 2 / 64, low 14 bits of the mantissa cleared
  constexpr double kLo = 2.572804622327669e-14;         // ln 2 / 64 - kHi
  constexpr double kMagic = 6755399441055744.0;         // 1.5 * 2^52: adds to an integer in the low word
  const double qc = NAN_SAFE ? (q > 800.0 ? 800.0 : q) : fmin(q, 800.0);
  const double t = fma(qc, -kInv, kMagic);
  const int n = __double2loint(t);
  const double k = t - kMagic;
  double r = fma(k, -kHi, -qc);
  r = fma(k, -kLo, r);
  double p = fma(r, 1.0 / 720.0, 1.0 / 120.0);
  p = fma(r, p, 1.0 / 24.0);
  p = fma(r, p, 1.0 / 6.0);
  p = fma(r, p, 0.5);
  p = fma(r, p, 1.0);
  const double e = exp_table()[n & ((1 << kExpBits) - 1)];
  return ldexp(fma(e * r, p, e), n >> kExpBits);
}

// log x for positive normal x: x = 2^e m with m in [0.70, 1.41), m c_i = 1 + r with
// |r| < 2^-7 next to 1 and 2^-8 elsewhere, log x = e ln 2 - log c_i + log1p r, the
// last through r^8 (first dropped term 1e-18 relative).  Within 2 ulp; 14 FP64 and 6
// integer instructions against about 30 for the atanh series that it replaces.
// NaN and infinities give NaN; zero a finite value: the pair sums only meet it in the
// self pair, which they discard.
__device__ __forceinline__ double log_fp64(double x) {
  constexpr double kLn2 = 0.69314718055994530942;
  const unsigned hi = (unsigned)__double2hiint(x);
  const int d = (int)(hi - kLogLow);
  const int e = d >> 20;
  const LogEntry t = log_table()[(d >> (20 - kLogBits)) & ((1 << kLogBits) - 1)];
  const double m = __hiloint2double((int)(hi - (unsigned)(d & ~0xfffff)), __double2loint(x));
  const double r = fma(m, t.c, -1.0);
  const double r2 = r * r;
  double p = fma(r, -1.0 / 8.0, 1.0 / 7.0);
  p = fma(r, p, -1.0 / 6.0);
  p = fma(r, p, 1.0 / 5.0);
  p = fma(r, p, -1.0 / 4.0);
  p = fma(r, p, 1.0 / 3.0);
  p = fma(r, p, -0.5);
  const double base = fma((double)e, kLn2, t.l);
  return fma(x, 0.0, base + fma(r2, p, r));
}
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }

// ---------------------------------------------------------------- policies
// A policy splits one pair into three phases so that the kernel can issue the
// phase for all R targets of a lane back to back (independent instruction
// streams hide the latency of the transcendental unit):
//   arg   : differences and the argument of the transcendental (kept in W)
//   trans : the one transcendental per pair (rcp, exp2 or log2)
//   acc   : weight and accumulate into NOUT tile partials
// W holds a policy's per-pair temporaries.

template <typename T>
struct W4 {
  T a, b, c, z;
};

template <typename T, bool USE_E>
struct SphereBS {
  static constexpr int NOUT = 3;
  static constexpr int IDX = 5;
  static constexpr int NW = SREC;
  static constexpr int TABLE = kNoTable;
  // acc += s * (x_i - y_j),  s = w2 / (|x_i - y_j|^2 + e_i + e_j); with
  // USE_E == false the points are on the sphere and e_i = e_j = 0.
  __device__ __forceinline__ static void arg(const Vec4<T>& t, const T* s, W4<T>& w) {
    w.a = t.a - s[0];
    w.b = t.b - s[1];
    w.c = t.c - s[2];
    T r2;
    if constexpr (USE_E)
      r2 = fma(w.a, w.a, t.d + s[3]);
    else
      r2 = w.a * w.a;
    r2 = fma(w.b, w.b, r2);
    w.z = fma(w.c, w.c, r2);
  }
  __device__ __forceinline__ static T trans(const W4<T>& w) {
    if constexpr (sizeof(T) == 4)
      return fast_rcp(w.z);
    else
      return rcp_refined(w.z);
  }
  __device__ __forceinline__ static void acc(const T* s, const W4<T>& w, T f, T a[NOUT]) {
    T q = s[4] * f;
    a[0] = fma(q, w.a, a[0]);
    a[1] = fma(q, w.b, a[1]);
    a[2] = fma(q, w.c, a[2]);
  }
};

template <typename T>
struct PlaneBS {
  static constexpr int NOUT = 2;
  static constexpr int IDX = 3;
  static constexpr int NW = SREC;
  static constexpr int TABLE = kNoTable;
  __device__ __forceinline__ static void arg(const Vec4<T>& t, const T* s, W4<T>& w) {
    w.a = t.a - s[0];
    w.b = t.b - s[1];
    w.z = fma(w.a, w.a, w.b * w.b);
  }
  __device__ __forceinline__ static T trans(const W4<T>& w) {
    if constexpr (sizeof(T) == 4)
      return fast_rcp(w.z);
    else
      return rcp_refined(w.z);
  }
  __device__ __forceinline__ static void acc(const T* s, const W4<T>& w, T f, T a[NOUT]) {
    T q = s[2] * f;
    a[0] = fma(q, w.b, a[0]);
    a[1] = fma(q, w.a, a[1]);
  }
};

// PSE Laplacian.  FP32: coordinates are pre-scaled by sqrt(log2 e)/eps so that
// q' = |dx|^2 = log2(e) rho^2, exp(-rho^2) = exp2(-q'), and the polynomial is
// re-expressed in q'.  FP64: coordinates scaled by 1/eps, q = rho^2.
template <typename T, int ORDER>
struct PsePolicy {
  static constexpr int NOUT = 1;
  static constexpr int IDX = 4;
  static constexpr int NW = SREC;
  static constexpr int TABLE = sizeof(T) == 8 ? kExpTable : kNoTable;
  __device__ __forceinline__ static void arg(const Vec4<T>& t, const T* s, W4<T>& w) {
    T dx = t.a - s[0], dy = t.b - s[1];
    w.z = fma(dx, dx, dy * dy);
    w.a = fma(-t.c, s[3], s[2]);  // f_j A_j - f_i A_j
  }
  __device__ __forceinline__ static T trans(const W4<T>& w) {
    if constexpr (sizeof(T) == 4)
      return fast_exp2(-w.z);
    else
      return exp_neg_fp64<ORDER == 2>(w.z);
  }
  __device__ __forceinline__ static void acc(const T* s, const W4<T>& w, T e, T a[NOUT]) {
    if constexpr (ORDER == 8) {
      // 40 - 40 rho^2 + 10 rho^4 - (2/3) rho^6 in the (scaled) variable q
      constexpr double L = sizeof(T) == 4 ? 1.4426950408889634 : 1.0;
      const T c0 = (T)40.0, c1 = (T)(-40.0 / L), c2 = (T)(10.0 / (L * L)),
              c3 = (T)(-(2.0 / 3.0) / (L * L * L));
      const T q = w.z;
      T p = fma(fma(fma(c3, q, c2), q, c1), q, c0);
      a[0] = fma(p * e, w.a, a[0]);
    } else {
      a[0] = fma(e, w.a, a[0]);
    }
  }
};

// Sphere PSE Laplacian (PSEDirectSum.f90:502-532): K8 of the great-circle
// distance R theta between the directions of x_i and x_j (SphereGeometry.f90:
// atan2(|x_i x x_j|, x_i . x_j) R).  Records hold the unit directions scaled by
// k R (k = sqrt(log2 e) / eps in FP32, 1 / eps in FP64), so that with
// u = |x'_i - x'_j|^2 / (k R)^2 = (c / R)^2 (c the chord) the scaled squared
// distance is q = (k R)^2 theta^2, theta = 2 asin(sqrt(u) / 2).
// SERIES: theta^2 = u g(u), g = sum_n a_n u^(n-1), a_n = 2 / (n^2 binom(2n, n))
// (the Taylor series of 4 asin^2(s / 2)), through n = SERIES; 0: by asin and sqrt.
// The caller takes the fewest terms that reach 7 eps (series_terms): in FP32 7 terms
// to 0.56 R and 14 to 1.2 R (first dropped term below 4e-9 relative), in FP64 10 to
// 0.35 R, 16 to 0.70 R and 28 to 1.16 R (2e-17).  Pairs farther than 7 eps get a
// slightly low theta^2, but their kernel factor exp(-q) is below e^-49.  The FP64
// gradient at level 6 (7 eps = 0.40 R) took 39.3 ms over all pairs by asin, 15.1 ms by
// 16 terms and the table exponential.
// Source record: {x', y', z', f A, A, idx, 1/(kR)^2, (kR)^2}; target {x', y', z', f}.
// Scaled squared great-circle distance q = (k R theta)^2 from the squared
// chord c2 = |x'_i - x'_j|^2 of directions scaled by k R; inv = 1/(k R)^2,
// kr2 = (k R)^2.
// Coefficient a_n of theta^2 = u g(u), g = sum a_n u^(n-1).
constexpr double theta2_coef(int n) {
  double a = 1.0;
  for (int k = 1; k < n; ++k) a *= (double)k * k / ((2.0 * k + 2.0) * (2.0 * k + 1.0));
  return a;
}

template <typename T, int SERIES>
__device__ __forceinline__ T sphere_q(T c2, T inv, T kr2) {
  const T u = c2 * inv;
  if constexpr (SERIES > 0) {
    T g = (T)theta2_coef(SERIES);
#pragma unroll
    for (int n = SERIES - 1; n >= 1; --n) g = fma(u, g, (T)theta2_coef(n));
    return c2 * g;
  } else {
    const T th = (T)2.0 * asin(fmin((T)0.5 * sqrt(u), (T)1.0));
    return th * th * kr2;
  }
}

template <typename T, int SERIES>
struct PseSphere {
  static constexpr int NOUT = 1;
  static constexpr int IDX = 5;
  static constexpr int NW = SREC;
  static constexpr int TABLE = sizeof(T) == 8 ? kExpTable : kNoTable;
  __device__ __forceinline__ static void arg(const Vec4<T>& t, const T* s, W4<T>& w) {
    const T dx = t.a - s[0], dy = t.b - s[1], dz = t.c - s[2];
    const T c2 = fma(dx, dx, fma(dy, dy, dz * dz));
    w.z = sphere_q<T, SERIES>(c2, s[6], s[7]);
    w.a = fma(-t.d, s[4], s[3]);  // f_j A_j - f_i A_j
  }
  __device__ __forceinline__ static T trans(const W4<T>& w) { return PsePolicy<T, 8>::trans(w); }
  __device__ __forceinline__ static void acc(const T* s, const W4<T>& w, T e, T a[NOUT]) {
    PsePolicy<T, 8>::acc(s, w, e, a);
  }
};

template <typename T, bool USE_E>
struct SphereGreen {
  static constexpr int NOUT = 2;
  static constexpr int IDX = 6;
  static constexpr int NW = SREC;
  static constexpr int TABLE = sizeof(T) == 8 ? kLogTable : kNoTable;
  __device__ __forceinline__ static void arg(const Vec4<T>& t, const T* s, W4<T>& w) {
    T dx = t.a - s[0], dy = t.b - s[1], dz = t.c - s[2];
    T r2;
    if constexpr (USE_E)
      r2 = fma(dx, dx, t.d + s[3]);
    else
      r2 = dx * dx;
    r2 = fma(dy, dy, r2);
    w.z = fma(dz, dz, r2);
  }
  __device__ __forceinline__ static T trans(const W4<T>& w) {
    if constexpr (sizeof(T) == 4)
      return fast_log2(w.z);  // log2(2 (R^2 - x.y))
    else
      return log_fp64((T)0.5 * w.z);  // ln(R^2 - x.y)
  }
  __device__ __forceinline__ static void acc(const T* s, const W4<T>& w, T lg, T a[NOUT]) {
    a[0] = fma(lg, s[4], a[0]);
    a[1] = fma(lg, s[5], a[1]);
  }
};

template <typename T>
struct PlaneGreen {
  static constexpr int NOUT = 1;
  static constexpr int IDX = 3;
  static constexpr int NW = SREC;
  static constexpr int TABLE = sizeof(T) == 8 ? kLogTable : kNoTable;
  __device__ __forceinline__ static void arg(const Vec4<T>& t, const T* s, W4<T>& w) {
    T dx = t.a - s[0], dy = t.b - s[1];
    w.z = fma(dx, dx, dy * dy);
  }
  __device__ __forceinline__ static T trans(const W4<T>& w) {
    if constexpr (sizeof(T) == 4)
      return fast_log2(w.z);
    else
      return log_fp64(w.z);
  }
  __device__ __forceinline__ static void acc(const T* s, const W4<T>& w, T lg, T a[NOUT]) {
    a[0] = fma(lg, s[2], a[0]);
  }
};

// Polynomial parts of the 8th-order PSE kernels in the scaled variable q
// (q = rho^2 in FP64, log2(e) rho^2 in FP32, where exp(-rho^2) = exp2(-q)):
//   derivative kernel (PSEDirectSum.f90:629-634): -20 + 20 r^2 - 5 r^4 + r^6/3
//   delta kernel      (PSEDirectSum.f90:611-616):   4 -  6 r^2 + 2 r^4 - r^6/6
//   Laplacian kernel  (PSEDirectSum.f90:622-627):  40 - 40 r^2 + 10 r^4 - 2 r^6/3
template <typename T>
__device__ __forceinline__ T cubic_in_q(T q, double c0, double c1, double c2, double c3) {
  constexpr double L = sizeof(T) == 4 ? 1.4426950408889634 : 1.0;
  return fma(fma(fma((T)(c3 / (L * L * L)), q, (T)(c2 / (L * L))), q, (T)(c1 / L)), q, (T)c0);
}

template <typename T>
__device__ __forceinline__ T exp_neg_q(T q) {
  if constexpr (sizeof(T) == 4)
    return fast_exp2(-q);
  else
    return exp_neg_fp64(q);
}

// PSE first-derivative sums (PSEDirectSum.f90:180-418, 537-579).  For M source
// fields c_m and the D coordinates of the separation X = x_i - x_j:
//   a[k]             = sum_j X_k K1'(q) A_j           (k < D)
//   a[D + m D + k]   = sum_j X_k K1'(q) c_m,j A_j
// (K1' the unnormalised kernel, coordinates scaled by sigma).  Every
// reference operator is an FP64 epilogue of these sums, since
// sum (c_j + c_i) X K1 A = a[D + m D + k] + c_i a[k].
// Source record: plane {x', y', A, c_0 .. c_{M-1}, idx};
// sphere {x', y', z', A, c_0 .., idx, 1/(kR)^2, (kR)^2} with x' the unit
// direction times k R (the separation is taken as R (d_i - d_j)).
template <typename T, bool SPH, int M, int SERIES>
struct PseDeriv {
  static constexpr int D = SPH ? 3 : 2;
  static constexpr int NOUT = D * (M + 1);
  static constexpr int IA = D;
  static constexpr int IC = D + 1;
  static constexpr int IDX = D + 1 + M;
  static constexpr int IINV = IDX + 1;
  static constexpr int IKR2 = IDX + 2;
  static constexpr int NW = (SPH ? IKR2 + 1 : IDX + 1) <= SREC ? SREC : SREC_MAX;
  static constexpr int TABLE = sizeof(T) == 8 ? kExpTable : kNoTable;
  static_assert((SPH ? IKR2 + 1 : IDX + 1) <= SREC_MAX, "record too long");
  __device__ __forceinline__ static void arg(const Vec4<T>& t, const T* s, W4<T>& w) {
    w.a = t.a - s[0];
    w.b = t.b - s[1];
    if constexpr (SPH) {
      w.c = t.c - s[2];
      const T c2 = fma(w.a, w.a, fma(w.b, w.b, w.c * w.c));
      w.z = sphere_q<T, SERIES>(c2, s[IINV], s[IKR2]);
    } else {
      w.z = fma(w.a, w.a, w.b * w.b);
    }
  }
  __device__ __forceinline__ static T trans(const W4<T>& w) { return exp_neg_q(w.z); }
  __device__ __forceinline__ static void acc(const T* s, const W4<T>& w, T e, T a[NOUT]) {
    const T g = cubic_in_q(w.z, -20.0, 20.0, -5.0, 1.0 / 3.0) * e * s[IA];
    T X[D];
    X[0] = w.a * g;
    X[1] = w.b * g;
    if constexpr (SPH) X[2] = w.c * g;
#pragma unroll
    for (int k = 0; k < D; ++k) {
      a[k] += X[k];
#pragma unroll
      for (int m = 0; m < M; ++m) a[D + m * D + k] = fma(s[IC + m], X[k], a[D + m * D + k]);
    }
  }
};

// PSE interpolation (PSEDirectSum.f90:121-168): sum_j f_j A_j Kd'(q).
// Source record: plane {x', y', f A, idx}; sphere {x', y', z', f A, idx,
// 1/(kR)^2, (kR)^2}.
template <typename T, bool SPH, int SERIES>
struct PseInterp {
  static constexpr int D = SPH ? 3 : 2;
  static constexpr int NOUT = 1;
  static constexpr int IFA = D;
  static constexpr int IDX = D + 1;
  static constexpr int NW = SREC;
  static constexpr int TABLE = sizeof(T) == 8 ? kExpTable : kNoTable;
  __device__ __forceinline__ static void arg(const Vec4<T>& t, const T* s, W4<T>& w) {
    const T dx = t.a - s[0], dy = t.b - s[1];
    if constexpr (SPH) {
      const T dz = t.c - s[2];
      w.z = sphere_q<T, SERIES>(fma(dx, dx, fma(dy, dy, dz * dz)), s[IDX + 1], s[IDX + 2]);
    } else {
      w.z = fma(dx, dx, dy * dy);
    }
  }
  __device__ __forceinline__ static T trans(const W4<T>& w) { return exp_neg_q(w.z); }
  __device__ __forceinline__ static void acc(const T* s, const W4<T>& w, T e, T a[NOUT]) {
    a[0] = fma(cubic_in_q(w.z, 4.0, -6.0, 2.0, -1.0 / 6.0) * e, s[IFA], a[0]);
  }
};

// Planar shallow-water right-hand side (SWEPlaneSolver.f90:457-538), one pass
// over the pairs for five sums: velocity (u, v) and its x derivative (ux, vx) of
// the point vortices and sources, and the K8 Laplacian of the surface height
// s = h + bottom (LAP; left out where its kernel is zero).
// Source record {x, y, a, b, s A, A, idx, c}: a = zeta A / (2 pi),
// b = delta A / (2 pi), c = log2(e) / eps^2 (FP32) or 1 / eps^2 (FP64).
// Target record {x, y, s, .}.  With f = 1 / r^2, p = (X b - Y a) f, q = (Y b + X a) f:
//   u  += p                      v  += q
//   ux += f (b - 2 X p)          vx += f (a - 2 X q)
//   lap += K8'(r^2 c) (s_j - s_i) A_j
// The flow of a pair is analytic away from its source, so uy = vx and vy = -ux
// for every pair and two of the four gradient sums are enough: 18 instructions
// per pair without the Laplacian against 35 for seven sums with it.
template <typename T, bool LAP = true>
struct SwePlane {
  static constexpr int NOUT = 5;
  static constexpr int IDX = 6;
  static constexpr int NW = SREC;
  static constexpr int TABLE = sizeof(T) == 8 ? kExpTable : kNoTable;
  __device__ __forceinline__ static void arg(const Vec4<T>& t, const T* s, W4<T>& w) {
    w.a = t.a - s[0];
    w.b = t.b - s[1];
    w.z = fma(w.a, w.a, w.b * w.b);
    if constexpr (LAP) w.c = fma(-t.c, s[5], s[4]);  // (s_j - s_i) A_j
  }
  __device__ __forceinline__ static T trans(const W4<T>& w) {
    if constexpr (sizeof(T) == 4)
      return fast_rcp(w.z);
    else
      return rcp_refined(w.z);
  }
  __device__ __forceinline__ static void acc(const T* s, const W4<T>& w, T f, T a[NOUT]) {
    const T X = w.a, Y = w.b;
    const T p = fma(X, s[3], -Y * s[2]) * f;
    const T q = fma(Y, s[3], X * s[2]) * f;
    const T X2 = X + X;
    a[0] += p;
    a[1] += q;
    a[2] = fma(f, fma(-X2, p, s[3]), a[2]);
    a[3] = fma(f, fma(-X2, q, s[2]), a[3]);
    if constexpr (LAP) {
      const T qq = w.z * s[7];
      a[4] = fma(cubic_in_q(qq, 40.0, -40.0, 10.0, -2.0 / 3.0) * exp_neg_q(qq), w.c, a[4]);
    }
  }
};

// ----------------------------------------------------------- the kernel
struct PairArgs {
  const void* tgt;   // nt target records (TREC words each)
  const void* src;   // ns source records (P::NW words each)
  double* partial;   // [nsplit][NOUT][nt]
  int nt;            // number of targets
  int tgt_idx0;      // particle index of target 0 (self-pair exclusion)
  int ns;            // number of sources
  int chunk;         // sources per split (multiple of kt)
  int nsplit;
  int kt;            // sources per compensated tile
  int n_wtiles;      // wave target tiles = ceil(nt / (64 R))
  // when set, the number of sources is read here and ns is only the bound
  // that sized chunk * nsplit (splits past the count sum nothing)
  const int* ns_dev = nullptr;
  float reach = 0.f;  // far path, shallow water: separation beyond which the exponential is zero
};

template <typename T>
__device__ __forceinline__ int rec_index(const T* s, int slot) {
  if constexpr (sizeof(T) == 4)
    return __float_as_int(s[slot]);
  else
    return (int)s[slot];
}

// Error-free (sum, compensation) update with a tile partial p.
template <typename T>
__device__ __forceinline__ void two_sum_acc(T& S, T& C, T p) {
  T t = S + p;
  T bp = t - S;
  T e = (S - (t - bp)) + (p - bp);
  C += e;
  S = t;
}

// Sources loaded together: 4 for the FP64 vortex sums (10-12 SGPRs a source), which
// took the level-4 sphere sum from 82 to 62 us and none slower at full size; the FP32
// sums and the longer PSE policies lose 5-35 % with 2 or 4 there and keep one ahead.
template <class P, typename T>
inline constexpr int LOAD_GROUP = 1;
template <bool E>
inline constexpr int LOAD_GROUP<SphereBS<double, E>, double> = 4;
template <bool E>
inline constexpr int LOAD_GROUP<SphereGreen<double, E>, double> = 4;
template <>
inline constexpr int LOAD_GROUP<PlaneBS<double>, double> = 4;
template <>
inline constexpr int LOAD_GROUP<PlaneGreen<double>, double> = 4;
// FP64 Biot-Savart sums take the reciprocals of a load group together (never of two
// targets: a value that is not finite stays with its target).  Kernels at icosahedral
// L4 / L5 / L6: 39.5 / 410 / 5,100 us one by one, 37 / 355 / 4,500 in fours; plane 300^2
// 3,280 / 2,720.  With R targets a lane the groups are kept apart by a scheduling
// barrier: interleaved they took 120 registers at R = 2, 86 apart, and 3 % longer.
template <class P, typename T>
inline constexpr bool RCP_FOUR = false;
template <bool E>
inline constexpr bool RCP_FOUR<SphereBS<double, E>, double> = true;
template <>
inline constexpr bool RCP_FOUR<PlaneBS<double>, double> = true;

// One wavefront's work: targets [t_begin, t_begin + 64 R) of the record array
// tg[0, nt) (particle index tgt_idx0 + local) against sources [j_begin, j_end)
// of src; FP64 results go to out[k * out_stride + i] for valid targets i.
// FOUR: reciprocals in fours; sums that are not finite are taken again without.
template <class P, typename T, int R, bool COMPENSATED, bool FOUR = RCP_FOUR<P, T>>
__device__ __forceinline__ void pair_tile(const Vec4<T>* __restrict__ tg, int nt, int t_begin,
                                          int tgt_idx0, const T* __restrict__ src, int j_begin,
                                          int j_end, int kt, double* __restrict__ out,
                                          int out_stride) {
  constexpr int NO = P::NOUT;
  const int lane = threadIdx.x & 63;
  Vec4<T> t[R];
  int tid[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    int i = t_begin + r * 64 + lane;
    int ic = i < nt ? i : nt - 1;
    t[r] = tg[ic];
    tid[r] = tgt_idx0 + i;
  }
  const int wt_lo = tgt_idx0 + t_begin;
  const int wt_hi = wt_lo + 64 * R - 1;

  T S[R][NO], C[R][NO];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int k = 0; k < NO; ++k) {
      S[r][k] = (T)0;
      C[r][k] = (T)0;
    }

  for (int jt = j_begin; jt < j_end; jt += kt) {
    const int jt_end = min(j_end, jt + kt);
    const int idx_lo = rec_index(src + (size_t)jt * P::NW, P::IDX);
    const int idx_hi = rec_index(src + (size_t)(jt_end - 1) * P::NW, P::IDX);
    const bool checked = (idx_lo <= wt_hi) && (idx_hi >= wt_lo);
    T p[R][NO];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int k = 0; k < NO; ++k) p[r][k] = (T)0;

    if (!checked) {
      // LOAD_GROUP sources' records load (scalar) under the arithmetic of the group
      // before them.  A record that another XCD packed takes 700 cycles, so where few
      // waves share a SIMD one record ahead leaves the loop waiting for each load.
      constexpr int G = LOAD_GROUP<P, T>;
      int j = jt;
      if (jt + G <= jt_end) {
        T sv[G][P::NW];
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int q = 0; q < P::NW; ++q) sv[g][q] = src[(size_t)(jt + g) * P::NW + q];
#pragma unroll 2
        for (; j + G <= jt_end; j += G) {
          const int jn = j + 2 * G <= jt_end ? j + G : j;
          T sn[G][P::NW];
#pragma unroll
          for (int g = 0; g < G; ++g)
#pragma unroll
            for (int q = 0; q < P::NW; ++q) sn[g][q] = src[(size_t)(jn + g) * P::NW + q];
          if constexpr (FOUR) {
            static_assert(G == 4);
#pragma unroll
            for (int r = 0; r < R; ++r) {
              W4<T> w[G];
              T z[G], f[G];
#pragma unroll
              for (int g = 0; g < G; ++g) {
                P::arg(t[r], sv[g], w[g]);
                z[g] = w[g].z;
              }
              rcp_four(z, f);
#pragma unroll
              for (int g = 0; g < G; ++g) P::acc(sv[g], w[g], f[g], p[r]);
              if (r + 1 < R) __builtin_amdgcn_sched_barrier(0);
            }
          } else {
#pragma unroll
            for (int g = 0; g < G; ++g) {
              W4<T> w[R];
              T f[R];
#pragma unroll
              for (int r = 0; r < R; ++r) P::arg(t[r], sv[g], w[r]);
#pragma unroll
              for (int r = 0; r < R; ++r) f[r] = P::trans(w[r]);
#pragma unroll
              for (int r = 0; r < R; ++r) P::acc(sv[g], w[r], f[r], p[r]);
            }
          }
#pragma unroll
          for (int g = 0; g < G; ++g)
#pragma unroll
            for (int q = 0; q < P::NW; ++q) sv[g][q] = sn[g][q];
        }
      }
      for (; j < jt_end; ++j) {
        T sv[P::NW];
#pragma unroll
        for (int q = 0; q < P::NW; ++q) sv[q] = src[(size_t)j * P::NW + q];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          W4<T> w;
          P::arg(t[r], sv, w);
          P::acc(sv, w, P::trans(w), p[r]);
        }
      }
    } else {
      for (int j = jt; j < jt_end; ++j) {
        const T* s = src + (size_t)j * P::NW;
        T sv[P::NW];
#pragma unroll
        for (int q = 0; q < P::NW; ++q) sv[q] = s[q];
        const int sidx = rec_index(sv, P::IDX);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          W4<T> w;
          P::arg(t[r], sv, w);
          T f = P::trans(w);
          T tmp[NO];
#pragma unroll
          for (int k = 0; k < NO; ++k) tmp[k] = (T)0;
          P::acc(sv, w, f, tmp);
          const bool self = (sidx == tid[r]);
#pragma unroll
          for (int k = 0; k < NO; ++k) p[r][k] += self ? (T)0 : tmp[k];
        }
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int k = 0; k < NO; ++k) {
        if constexpr (COMPENSATED)
          two_sum_acc(S[r][k], C[r][k], p[r][k]);
        else
          S[r][k] += p[r][k];
      }
  }

  if constexpr (FOUR) {
    bool bad = false;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int k = 0; k < NO; ++k) bad = bad || !__builtin_isfinite(S[r][k]);
    if (__any(bad)) {
      pair_tile<P, T, R, COMPENSATED, false>(tg, nt, t_begin, tgt_idx0, src, j_begin, j_end, kt, out, out_stride);
      return;
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    int i = t_begin + r * 64 + lane;
    if (i < nt) {
#pragma unroll
      for (int k = 0; k < NO; ++k) out[(size_t)k * out_stride + i] = (double)S[r][k] + (double)C[r][k];
    }
  }
}

template <class P, typename T, int R, bool COMPENSATED>
__global__ __launch_bounds__(256) void pair_sum_kernel(PairArgs a) {
  fill_tables<P::TABLE>();
  const int wid = threadIdx.x >> 6;
  const int nblk_t = (a.n_wtiles + 3) >> 2;
  const int split = blockIdx.x / nblk_t;
  const int wtile = (blockIdx.x - split * nblk_t) * 4 + wid;
  if (wtile >= a.n_wtiles) return;  // wave-uniform
  const int ns = a.ns_dev ? *a.ns_dev : a.ns;
  const int j_begin = split * a.chunk;
  const int j_end = min(ns, j_begin + a.chunk);
  pair_tile<P, T, R, COMPENSATED>(reinterpret_cast<const Vec4<T>*>(a.tgt), a.nt, wtile * 64 * R,
                                  a.tgt_idx0, reinterpret_cast<const T*>(a.src), j_begin, j_end, a.kt,
                                  a.partial + (size_t)split * P::NOUT * a.nt, a.nt);
}

// ------------------------------------------------------- batched problems
// Many independent problems in one persistent launch.  Problem k owns target
// records [t_off, t_off + nt) (particle indices t_off + local), source records
// [s_off, s_off + ns) and FP64 partials at part_off ([nsplit][NOUT][nt]).
// A work item is (problem, wave target tile, source split); items are taken
// from a device counter by whole wavefronts until the list is exhausted, so
// every wave reaches the exit.
struct BatchProblem {
  int t_off, nt, s_off, ns;
  int chunk, nsplit;
  long long part_off;
  int far;                   // takes the far path (far_kernels.hpp)
  int tball_off, sball_off;  // its balls
};

struct BatchItem {
  int prob, wtile, split, pad;
};

struct BatchArgs {
  const void* tgt;
  const void* src;
  double* partial;
  const BatchProblem* probs;
  const BatchItem* items;
  int n_items;
  int kt;
  unsigned int* counter;
};

// The buffers are separate __restrict__ kernel parameters rather than fields
// of BatchArgs: the loop stores partials and then reads sources of the next
// item, and only kernel-level noalias lets the compiler keep the source reads
// on the scalar unit (wave-uniform s_load, SGPR operands) across those stores.
// Through a struct, it issued per-lane vector loads of the same addresses.
// Waves a SIMD must hold: 6 in FP32; FP64 at the registers its reciprocals in fours
// take without spills (86, 166 and 256 at R = 2, 4 and 8).
template <typename T, int R>
inline constexpr int batch_waves = sizeof(T) == 4 || R == 1 ? 6 : R == 2 ? 5 : R == 4 ? 3 : 1;
template <class P, typename T, int R, bool COMPENSATED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(batch_waves<T, R>))) void pair_batch_kernel(
    const void* __restrict__ tgt, const void* __restrict__ srcv, double* __restrict__ partial,
    const BatchProblem* __restrict__ probs, const BatchItem* __restrict__ items, int n_items, int kt,
    unsigned int* __restrict__ counter) {
  const int lane = threadIdx.x & 63;
  const Vec4<T>* tg = reinterpret_cast<const Vec4<T>*>(tgt);
  const T* src = reinterpret_cast<const T*>(srcv);
  for (;;) {
    int item = 0;
    if (lane == 0) item = (int)atomicAdd(counter, 1u);
    item = __builtin_amdgcn_readfirstlane(__shfl(item, 0));
    if (item >= n_items) break;
    const BatchItem it = items[item];
    const BatchProblem pr = probs[it.prob];
    const int j_begin = pr.s_off + it.split * pr.chunk;
    const int j_end = min(pr.s_off + pr.ns, j_begin + pr.chunk);
    pair_tile<P, T, R, COMPENSATED>(tg + pr.t_off, pr.nt, it.wtile * 64 * R, pr.t_off, src, j_begin, j_end,
                                    kt, partial + pr.part_off + (size_t)it.split * P::NOUT * pr.nt, pr.nt);
  }
}

}  // namespace lpm
