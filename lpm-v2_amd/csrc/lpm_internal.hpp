// lpm_internal.hpp -- context, device buffers and the pair-sum driver.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <vector>

#include "../../include/lpm_direct.h"

#define LPM_VERSION_NUMBER 10000

namespace lpm {

// Grow-only device buffer owned by a context or solver.  A `fixed` buffer is
// a view of memory owned elsewhere (a segment of the static scratch array):
// it never allocates or frees, and a request beyond its size fails.
struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  bool fixed = false;
  static DevBuf view(void* ptr, size_t n) {
    DevBuf b;
    b.p = ptr;
    b.bytes = n;
    b.fixed = true;
    return b;
  }
  hipError_t ensure(size_t n) {
    if (n <= bytes) return hipSuccess;
    if (fixed) return hipErrorOutOfMemory;
    if (p) {
      hipError_t e = hipFree(p);
      p = nullptr;
      bytes = 0;
      if (e != hipSuccess) return e;
    }
    hipError_t e = hipMalloc(&p, n < 256 ? 256 : n);
    if (e == hipSuccess) bytes = n < 256 ? 256 : n;
    return e;
  }
  void release() {
    if (p && !fixed) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  }
  template <typename T>
  T* as() const {
    return reinterpret_cast<T*>(p);
  }
};

struct Tuning {
  int r = 0;       // targets per lane
  int kt = 0;      // sources per compensated tile
  int splits = 0;  // 0 = automatic
};

struct EventPair {
  hipEvent_t a, b;
  int kind;
};

}  // namespace lpm

struct lpm_ctx {
  int device = 0;
  int num_cus = 256;
  hipStream_t stream = nullptr;
  std::string err;
  // stateless-call staging
  lpm::DevBuf in[12];
  lpm::DevBuf out[4];
  lpm::DevBuf list, flags;
  lpm::DevBuf stage;  // the staged calls' inputs and outputs (lpm_api.hip)
  void* pin = nullptr;  // pinned host block of the same size
  lpm::DevBuf tgt, src, partial;
  lpm::DevBuf red;  // reductions
  lpm::DevBuf order;  // spatial order of the tile paths
  // this device's copy of the static scratch array (lpm_api.hip), resolved
  // once at lpm_create; used by the allocation-free entry point only
  void* scratch = nullptr;
  // tuning per kind and precision
  lpm::Tuning tune[LPM_K_COUNT][2];
  // timing
  bool timing = false;
  std::vector<lpm::EventPair> pending;
  std::vector<hipEvent_t> event_pool;
  int64_t launches[LPM_K_COUNT] = {0};
  double total_ms[LPM_K_COUNT] = {0};
};

namespace lpm {

// Error helpers: every failing path records a message on the context.
int fail(lpm_ctx* ctx, int code, const std::string& msg);
int hip_fail(lpm_ctx* ctx, hipError_t e, const char* what);

#define LPM_HIP(ctx, expr)                                   \
  do {                                                       \
    hipError_t _e = (expr);                                  \
    if (_e != hipSuccess) return ::lpm::hip_fail(ctx, _e, #expr); \
  } while (0)

// Description of one all-pairs sum over device-resident FP64 inputs.
// Targets are particles [i0, i1) of the arrays; sources are the particles in
// `src_list` (device int array of ns particle indices, ascending).
struct PairProblem {
  int kind = LPM_K_SPHERE_BS;
  int precision = LPM_PREC_FP32_KAHAN;
  int n = 0;         // particles in the arrays
  int i0 = 0, i1 = 0;
  const double* x = nullptr;
  const double* y = nullptr;
  const double* z = nullptr;
  const double* q0 = nullptr;  // zeta_rel / omega / f
  const double* q1 = nullptr;  // zeta_abs (sphere stream)
  const double* area = nullptr;
  const int* src_list = nullptr;
  int ns = 0;
  const int* active = nullptr;  // device 0/1 flags (sphere stream self term)
  double radius = 1.0;
  bool on_sphere = false;  // all points on the sphere of `radius` (drop the R^2-|x|^2 terms)
  double eps = 1.0;
  double* out0 = nullptr;  // device outputs, indexed by particle (i0..i1-1)
  double* out1 = nullptr;
  double* out2 = nullptr;
  // PSE derivative / SWE kinds: more fields and outputs, the epilogue op and
  // the number of derivative fields m.
  const double* q2 = nullptr;
  const double* q3 = nullptr;
  double* out3 = nullptr;
  int op = 0;
  int m = 1;
  // Targets at points other than the particles (interpolation, Laplacian at
  // points): when tx is set, targets are tx/ty/tz[/tq][i0..i1), outputs are
  // indexed by point, and no self pair is excluded.
  const double* tx = nullptr;
  const double* ty = nullptr;
  const double* tz = nullptr;
  const double* tq = nullptr;
  // Optional caller-owned scratch; when null the context's buffers are used.
  DevBuf* tgt_buf = nullptr;
  DevBuf* src_buf = nullptr;
  DevBuf* partial_buf = nullptr;
  DevBuf* red_buf = nullptr;  // FP32 sphere Green: the two FP64 source totals and their partials
  DevBuf* order_buf = nullptr;
  // Spatial order of targets and sources when the caller has it (a solver keeps
  // one for the four sums of a step); else run_pair_sum makes one where it is used.
  const int* tgt_order = nullptr;
  const int* src_order = nullptr;
  // Plane PSE kinds: share of the pairs within kTestedReach eps, as far as the caller
  // knows it (see sum_path)
  double reach_share = 0.0;
  // Source count on the device (set by a device-side compaction): ns is then
  // an upper bound that sizes the launches, and the kernels read the count.
  // Such a sum also records no timing events.
  const int* ns_dev = nullptr;
};

// Epilogues of the PSE derivative kinds.
enum PseOp { kOpGradient = 0, kOpSecondPartials = 1, kOpDoubleDot = 2, kOpDivergence = 3 };

// Enqueue the whole sum (pack, pair kernel, finalize) on ctx->stream.
int run_pair_sum(lpm_ctx* ctx, const PairProblem& pp);

// Record packing (FP64 SoA -> FP32/FP64 pair records).  prad, when not null,
// gives a per-particle sphere radius (batched problems).
struct PackArgs {
  const double *x, *y, *z, *q0, *q1, *area;
  const double* prad;
  const int* list;
  int count;  // records to write
  int i0;     // first target particle (targets)
  double radius, sigma;
  const double* q2 = nullptr;
  const double* q3 = nullptr;
  int m = 1;        // derivative fields
  double aux = 0.0; // SWE: log2(e)/eps^2 (FP32) or 1/eps^2 (FP64)
  const int* count_dev = nullptr;  // sources: record count on the device (count is then a bound)
  const int* tgt_order = nullptr;  // targets: particle of every record (null: i0 + record)
};

// Ordered sum over source splits and the FP64 epilogue of one kind.
struct FinArgs {
  const double* partial;
  int nt, i0, nsplit;
  const double *x, *y, *z, *q0, *q1, *area;
  const int* active;
  const double* G;
  double radius, scale;
  int fp32;
  double *out0, *out1, *out2;
  const double* q2 = nullptr;
  double* out3 = nullptr;
  int op = 0;
  const int* tgt_order = nullptr;  // particle of every target record (null: i0 + record)
};

// The PSE derivative, interpolation and SWE kinds (lpm_pse_ops.hip).
bool is_ops_kind(int kind);
int ops_nout(int kind, int m);
int ops_record_words(int kind, int m);
// series: terms of the sphere distance series, 0 by asin
const void* ops_pick_kernel(int kind, int prec, int r, int m, int series);
const void* ops_pick_cull(int kind, int prec, int m, int series);
void ops_launch_pack(int kind, int prec, const PackArgs& s, const PackArgs& t, void* srec, void* trec, int ns,
                     int nt, hipStream_t st);
int ops_launch_finalize(int kind, int m, const FinArgs& f, hipStream_t st);
void launch_pack(int kind, int precision, const PackArgs& a, void* srec, void* trec, int ns, int nt,
                 hipStream_t st);
Tuning default_tuning(int kind, int prec);
// Where the far path starts, in pairs (see sum_path).
constexpr double kFarMinPairsSphere = 2e9, kFarMinPairsPlane = 4e9, kFarMinPairsSwe = 4e9;

// How a sum is scheduled: over all pairs (pair_kernels.hpp), with the
// well-separated tiles on the MFMA (far_kernels.hpp), or without the tiles whose
// terms are zero (cull_kernels.hpp).  The last two want the records in spatial order.
enum SumPath { kAllPairs = 0, kFarTiles = 1, kCullTiles = 2 };
// reach_share: of a PSE sum, the share of the pairs within kTestedReach eps
SumPath sum_path(const lpm_ctx* ctx, int kind, int prec, int nt, int ns, double reach_share = 0.0);
constexpr double kCullMinPairs = 1.5e8;
// The tested tiles leave about this reach, in eps, of the 10.2 (FP32) and 27.3 (FP64)
// at which terms are zero.
constexpr double kTestedReach = 8.5;

// Spatial order (lpm_order.hip) of targets tx.. [i0, i0 + nt) and of the sources
// x..[list[0, ns)]: device arrays of particle indices inside `buf`.
struct OrderInput {
  const double *tx, *ty, *tz;
  int i0, nt;
  const double *x, *y, *z;
  const int* list;
  int ns;
  bool sphere;
  // batched sphere problems, ordered problem by problem: the problem of every
  // particle, whether a problem is sorted at all, and the largest problem's size
  const int* prob = nullptr;
  const int* sorted = nullptr;
  int n_prob = 0, max_n = 0;
};
size_t order_bytes(int nt, int ns);  // spatial_order allocates nothing in a buffer of this size
int spatial_order(lpm_ctx* ctx, const OrderInput& in, DevBuf& buf, int** tgt_order, int** src_order);

// The same stable sort on n targets and n sources with keys of the caller's:
// `buf` holds cell_sort_bytes(n); fill the input, then sort by `bits` bits.
struct CellSort {
  unsigned *tgt_key, *src_key;
  int *tgt_val, *src_val;
};
size_t cell_sort_bytes(int n);
CellSort cell_sort_input(DevBuf& buf, int n);
void cell_sort(hipStream_t st, DevBuf& buf, int n, int bits, int* tgt_perm, int* src_perm, const unsigned** tgt_key,
               const unsigned** src_key);

int blocks_per_cu(const void* kernel);
hipEvent_t take_event(lpm_ctx* ctx);

// Resolve queued timing events (synchronizes the stream).
int collect_timing(lpm_ctx* ctx);

// FP64 reductions over active particles: {sum |u|^2 A, sum q^2 A, sum q A}.
int run_diagnostics(lpm_ctx* ctx, int n, const double* u, const double* v, const double* w,
                    const double* q, const double* area, const int* active, double out[3]);

// Active-particle list on the device from host flags (ascending indices), and the
// flags themselves (any nonzero value is true).
int upload_active_list(lpm_ctx* ctx, const int32_t* active_host, int n, DevBuf& list,
                       DevBuf* flags, int* ns_out);

}  // namespace lpm
