// lpm_order.hip -- spatial order of targets and sources.
//
// The tile paths (far_kernels.hpp, cull_kernels.hpp) decide per tile of consecutive
// records, so they want consecutive records close together, whatever order the
// caller's particles come in (row-major grids, mesh levels one after the other,
// remeshed sets).  Points are sorted by their index along a Hilbert curve: over the
// bounding box on the plane, over the six faces of the surrounding cube on the
// sphere.  Consecutive tiles are then compact patches for any input order.
//
// The sort is a stable least-significant-digit radix sort, 8 bits a pass: per-block
// digit counts, a scan per digit, stable scatter.  Targets and sources go through the same
// launches (two segments), three a pass beside the keys' one and, on the plane, the
// bounding box's: keys have 8-24 bits on the plane, 11-27 on the sphere and up to 32 in
// batches, 5-11 and 7-13 short launches for both.  It is deterministic, allocates nothing
// and holds no memset, so it may be captured.  rocPRIM's sort takes a merge-sort path of
// about 24 launches (130 us) at these sizes.
#include "lpm_internal.hpp"

namespace lpm {

namespace {

constexpr int kSortThreads = 256;
constexpr int kSortRounds = 8;                                // items per thread
constexpr int kSortItems = kSortThreads * kSortRounds;        // items per block
constexpr int kBins = 256;
constexpr int kBoxBlocks = 256;

// Index of cell (x, y) of the 2^k x 2^k grid along the Hilbert curve.
__device__ __forceinline__ unsigned hilbert(unsigned x, unsigned y, int k) {
  unsigned d = 0;
  for (int s = k - 1; s >= 0; --s) {
    const unsigned rx = (x >> s) & 1u, ry = (y >> s) & 1u;
    d = d * 4u + ((3u * rx) ^ ry);
    if (ry == 0u) {  // rotate the quadrant
      if (rx == 1u) {
        x = ~x;
        y = ~y;
      }
      const unsigned t = x;
      x = y;
      y = t;
    }
  }
  return d;
}

__device__ __forceinline__ unsigned cell_of(double u, int k) {  // u in [0, 1]
  const double c = u * (double)(1 << k);
  return (unsigned)fmin(fmax(c, 0.0), (double)((1 << k) - 1));  // NaN goes to cell 0
}

struct Segment {
  const double *x, *y, *z;
  const int* list;  // particle of item i, or null: i0 + i
  int i0, n;
};

struct OrderDev {
  Segment seg[2];
  int k;        // bits per coordinate
  int sphere;
  const double* box;  // plane: kBoxBlocks x {xmin, ymin, xmax, ymax}
  const int* prob;    // batched problems: the problem of a particle, above the curve index in the key
  const int* sorted;  // per problem: 0 keeps its particles in the caller's order
};

__device__ __forceinline__ int item_particle(const Segment& s, int i) { return s.list ? s.list[i] : s.i0 + i; }

// Plane: bounding box of both segments, one partial box per block.
__global__ __launch_bounds__(256) void box_partial(OrderDev a, double* __restrict__ box) {
  __shared__ double red[4][4];
  double lo[2] = {1e308, 1e308}, hi[2] = {-1e308, -1e308};
  const int total = a.seg[0].n + a.seg[1].n;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += kBoxBlocks * 256) {
    const bool second = i >= a.seg[0].n;
    const Segment& s = a.seg[second ? 1 : 0];
    const int p = item_particle(s, second ? i - a.seg[0].n : i);
    const double c[2] = {s.x[p], s.y[p]};
    for (int q = 0; q < 2; ++q) {
      if (!isfinite(c[q])) continue;
      lo[q] = fmin(lo[q], c[q]);
      hi[q] = fmax(hi[q], c[q]);
    }
  }
  for (int m = 32; m > 0; m >>= 1)
    for (int q = 0; q < 2; ++q) {
      lo[q] = fmin(lo[q], __shfl_xor(lo[q], m));
      hi[q] = fmax(hi[q], __shfl_xor(hi[q], m));
    }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[w][0] = lo[0], red[w][1] = lo[1], red[w][2] = hi[0], red[w][3] = hi[1];
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    const int q = threadIdx.x;
    double v = red[0][q];
    for (int j = 1; j < 4; ++j) v = q < 2 ? fmin(v, red[j][q]) : fmax(v, red[j][q]);
    box[blockIdx.x * 4 + q] = v;
  }
}

// Key of every item; items are laid out segment 0 first, then segment 1.
__global__ __launch_bounds__(256) void make_keys(OrderDev a, unsigned* __restrict__ keys, int* __restrict__ vals) {
  __shared__ double box[4];
  if (!a.sphere) {
    __shared__ double part[4][4];
    double v[4];
    for (int q = 0; q < 4; ++q) v[q] = a.box[threadIdx.x * 4 + q];
    for (int m = 32; m > 0; m >>= 1)
      for (int q = 0; q < 4; ++q) v[q] = q < 2 ? fmin(v[q], __shfl_xor(v[q], m)) : fmax(v[q], __shfl_xor(v[q], m));
    if ((threadIdx.x & 63) == 0)
      for (int q = 0; q < 4; ++q) part[threadIdx.x >> 6][q] = v[q];
    __syncthreads();
    if (threadIdx.x < 4) {
      const int q = threadIdx.x;
      double r = part[0][q];
      for (int w = 1; w < 4; ++w) r = q < 2 ? fmin(r, part[w][q]) : fmax(r, part[w][q]);
      box[q] = r;
    }
    __syncthreads();
  }
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.seg[0].n + a.seg[1].n) return;
  const bool second = i >= a.seg[0].n;
  const Segment& s = a.seg[second ? 1 : 0];
  const int p = item_particle(s, second ? i - a.seg[0].n : i);
  const double x = s.x[p], y = s.y[p];
  unsigned key;
  if (a.sphere) {
    const double z = s.z[p];
    const double ax = fabs(x), ay = fabs(y), az = fabs(z);
    // faces in the order +x +y +z -y -z -x, each entered at the corner where the
    // curve left the one before, so that no tile jumps across the sphere; u runs
    // along the edge from the entry to the exit corner
    double m, u, v;
    unsigned face;
    if (ax >= ay && ax >= az) {
      m = ax;
      if (x >= 0.0)
        face = 0u, u = -z, v = -y;
      else
        face = 5u, u = y, v = z;
    } else if (ay >= az) {
      m = ay;
      if (y >= 0.0)
        face = 1u, u = z, v = -x;
      else
        face = 3u, u = -z, v = -x;
    } else {
      m = az;
      if (z >= 0.0)
        face = 2u, u = -y, v = -x;
      else
        face = 4u, u = -x, v = y;
    }
    const double h = 0.5 / m;
    key = (face << (2 * a.k)) | hilbert(cell_of(0.5 + u * h, a.k), cell_of(0.5 + v * h, a.k), a.k);
    if (a.prob) {
      const int pr = a.prob[p];
      key = ((unsigned)pr << (2 * a.k + 3)) | (a.sorted[pr] ? key : 0u);
    }
  } else {
    // one scale for both coordinates, so that cells are square
    const double ext = fmax(box[2] - box[0], box[3] - box[1]);
    const double sc = ext > 0.0 ? 1.0 / ext : 0.0;
    key = hilbert(cell_of((x - box[0]) * sc, a.k), cell_of((y - box[1]) * sc, a.k), a.k);
  }
  keys[i] = key;
  vals[i] = p;
}

struct SortDev {
  int n0, n1;   // items per segment
  int b0, b1;   // blocks per segment
  int shift;
  const unsigned* kin;
  const int* vin;
  unsigned* kout;
  int* vout0;  // segment 0
  int* vout1;  // segment 1
  int* hist;   // [segment][bin][block]
  int* total;  // [segment][bin]
};

__device__ __forceinline__ void sort_segment(const SortDev& a, int& base, int& n, int& blk, int& nblk, int*& hist) {
  const bool second = (int)blockIdx.x >= a.b0;
  base = second ? a.n0 : 0;
  n = second ? a.n1 : a.n0;
  blk = second ? blockIdx.x - a.b0 : blockIdx.x;
  nblk = second ? a.b1 : a.b0;
  hist = a.hist + (second ? kBins * a.b0 : 0);
}

__global__ __launch_bounds__(kSortThreads) void sort_count(SortDev a) {
  __shared__ int cnt[kBins];
  int base, n, blk, nblk;
  int* hist;
  sort_segment(a, base, n, blk, nblk, hist);
  cnt[threadIdx.x] = 0;
  __syncthreads();
  for (int r = 0; r < kSortRounds; ++r) {
    const int i = blk * kSortItems + r * kSortThreads + threadIdx.x;
    if (i < n) atomicAdd(&cnt[(a.kin[base + i] >> a.shift) & (kBins - 1)], 1);
  }
  __syncthreads();
  hist[threadIdx.x * nblk + blk] = cnt[threadIdx.x];
}

// Exclusive scan of each bin's counts over the blocks (one block per segment and
// bin) and the bin's total; the scatter adds the totals of the bins before it.
__global__ __launch_bounds__(256) void sort_scan(SortDev a) {
  __shared__ int wsum[4];
  const bool second = blockIdx.x >= kBins;
  const int bin = blockIdx.x & (kBins - 1);
  const int nblk = second ? a.b1 : a.b0;
  int* h = a.hist + (second ? kBins * a.b0 : 0) + (size_t)bin * nblk;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int carry = 0;
  for (int b = 0; b < nblk; b += 256) {
    const int i = b + threadIdx.x;
    const int mine = i < nblk ? h[i] : 0;
    int inc = mine;
    for (int m = 1; m < 64; m <<= 1) {
      const int o = __shfl_up(inc, m);
      if (lane >= m) inc += o;
    }
    if (lane == 63) wsum[wid] = inc;
    __syncthreads();
    int before = carry, all = 0;
    for (int w = 0; w < 4; ++w) {
      const int s = wsum[w];
      if (w < wid) before += s;
      all += s;
    }
    if (i < nblk) h[i] = before + inc - mine;
    carry += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) a.total[blockIdx.x] = carry;
}

// Stable scatter.  A wave owns kSortItems / 4 consecutive items; within a round of
// 64 an item's rank among equal digits comes from 8 ballots.
__global__ __launch_bounds__(kSortThreads) void sort_scatter(SortDev a) {
  __shared__ int place[4][kBins];
  __shared__ int wsum[4];
  int base, n, blk, nblk;
  int* hist;
  sort_segment(a, base, n, blk, nblk, hist);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (int w = 0; w < 4; ++w) place[w][threadIdx.x] = 0;
  __syncthreads();
  const int first = blk * kSortItems + wid * (kSortItems / 4);
  unsigned key[kSortRounds];
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r) {
    const int i = first + r * 64 + lane;
    key[r] = i < n ? a.kin[base + i] : 0u;
    if (i < n) atomicAdd(&place[wid][(key[r] >> a.shift) & (kBins - 1)], 1);
  }
  // first place of this thread's bin: totals of the bins before it
  const int total = a.total[((int)blockIdx.x >= a.b0 ? kBins : 0) + threadIdx.x];
  int inc = total;
  for (int m = 1; m < 64; m <<= 1) {
    const int o = __shfl_up(inc, m);
    if (lane >= m) inc += o;
  }
  if (lane == 63) wsum[wid] = inc;
  __syncthreads();
  {
    int at = hist[threadIdx.x * nblk + blk] + inc - total;
    for (int w = 0; w < wid; ++w) at += wsum[w];
    for (int w = 0; w < 4; ++w) {
      const int c = place[w][threadIdx.x];
      place[w][threadIdx.x] = at;
      at += c;
    }
  }
  __syncthreads();
  int* vout = (int)blockIdx.x >= a.b0 ? a.vout1 : a.vout0;
  volatile int* mine = place[wid];  // read and written by different lanes of the wave in turn
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r) {
    const int i = first + r * 64 + lane;
    const bool in = i < n;
    const unsigned d = (key[r] >> a.shift) & (kBins - 1);
    unsigned long long same = __ballot(in);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const unsigned long long m = __ballot((d >> b) & 1u);
      same &= (d >> b) & 1u ? m : ~m;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull));
    int at = 0;
    if (in) at = mine[d] + rank;
    __builtin_amdgcn_wave_barrier();
    if (in && rank == 0) mine[d] = at + __popcll(same);
    __builtin_amdgcn_wave_barrier();
    if (in) {
      a.kout[base + at] = key[r];
      vout[at] = a.vin[base + i];
    }
  }
}

int sort_blocks(int n) { return (n + kSortItems - 1) / kSortItems; }
size_t up256(size_t b) { return (b + 255) / 256 * 256; }

// Buffers of a sort of n0 + n1 items, laid out from p.
struct SortSpace {
  unsigned* key[2];
  int* val[2];
  int *hist, *total;
};

SortSpace sort_space(char* p, int n0, int n1) {
  auto take = [&](size_t b) {
    char* r = p;
    p += up256(b);
    return r;
  };
  const size_t items = (size_t)n0 + n1;
  SortSpace w;
  for (int q = 0; q < 2; ++q) w.key[q] = reinterpret_cast<unsigned*>(take(items * 4));
  for (int q = 0; q < 2; ++q) w.val[q] = reinterpret_cast<int*>(take(items * 4));
  w.hist = reinterpret_cast<int*>(take(((size_t)sort_blocks(n0) + sort_blocks(n1)) * kBins * 4));
  w.total = reinterpret_cast<int*>(take(2 * kBins * 4));
  return w;
}

// Sort key[0], val[0] (segment 0, then segment 1) by `bits` bits; the values go to
// out0 and out1, the sorted keys to key[passes & 1].
const unsigned* sort_pairs(hipStream_t st, const SortSpace& w, int n0, int n1, int bits, int* out0, int* out1) {
  const int b0 = sort_blocks(n0), b1 = sort_blocks(n1);
  const int passes = (bits + 7) / 8;
  for (int q = 0; q < passes; ++q) {
    const bool last = q == passes - 1;
    SortDev s{n0, n1, b0, b1, 8 * q, w.key[q & 1], w.val[q & 1], w.key[(q + 1) & 1],
              last ? out0 : w.val[(q + 1) & 1], last ? out1 : w.val[(q + 1) & 1] + n0, w.hist, w.total};
    hipLaunchKernelGGL(sort_count, dim3(b0 + b1), dim3(kSortThreads), 0, st, s);
    hipLaunchKernelGGL(sort_scan, dim3(2 * kBins), dim3(256), 0, st, s);
    hipLaunchKernelGGL(sort_scatter, dim3(b0 + b1), dim3(kSortThreads), 0, st, s);
  }
  return w.key[passes & 1];
}

}  // namespace

size_t cell_sort_bytes(int n) {
  return 4 * up256(2 * (size_t)n * 4) + up256(2 * (size_t)sort_blocks(n) * kBins * 4) + up256(2 * kBins * 4);
}

CellSort cell_sort_input(DevBuf& buf, int n) {
  const SortSpace w = sort_space(buf.as<char>(), n, n);
  return CellSort{w.key[0], w.key[0] + n, w.val[0], w.val[0] + n};
}

void cell_sort(hipStream_t st, DevBuf& buf, int n, int bits, int* tgt_perm, int* src_perm, const unsigned** tgt_key,
               const unsigned** src_key) {
  const unsigned* k = sort_pairs(st, sort_space(buf.as<char>(), n, n), n, n, bits, tgt_perm, src_perm);
  *tgt_key = k;
  *src_key = k + n;
}

size_t order_bytes(int nt, int ns) {
  const size_t items = (size_t)nt + ns;
  const size_t blocks = (size_t)sort_blocks(nt) + sort_blocks(ns);
  return 4 * up256(items * 4) + up256(blocks * kBins * 4) + up256(2 * kBins * 4) + up256(kBoxBlocks * 4 * sizeof(double)) +
         up256((size_t)nt * 4) + up256((size_t)ns * 4);
}

int spatial_order(lpm_ctx* ctx, const OrderInput& in, DevBuf& buf, int** tgt_order, int** src_order) {
  LPM_HIP(ctx, buf.ensure(order_bytes(in.nt, in.ns)));
  const int items = in.nt + in.ns;
  char* p = buf.as<char>();
  auto take = [&](size_t b) {
    char* r = p;
    p += up256(b);
    return r;
  };
  // the results first: their place depends on nt and ns alone
  int* tout = reinterpret_cast<int*>(take((size_t)in.nt * 4));
  int* sout = reinterpret_cast<int*>(take((size_t)in.ns * 4));
  double* box = reinterpret_cast<double*>(take(kBoxBlocks * 4 * sizeof(double)));
  const SortSpace w = sort_space(p, in.nt, in.ns);
  *tgt_order = tout;
  *src_order = sout;
  if (items == 0) return LPM_OK;

  // about 8 points a cell: tiles hold 64-256, and fewer key bits save passes
  // (16 bits: 2 passes to 524,288 points on the plane, 196,608 on the sphere)
  const int n = in.prob ? in.max_n : in.nt > in.ns ? in.nt : in.ns;
  int prob_bits = 0;
  if (in.prob)
    while ((1 << prob_bits) < in.n_prob) ++prob_bits;
  int k = 4;
  while (k < 12 && 2 * (k + 1) + 3 + prob_bits <= 32 && ((long long)(in.sphere ? 6 : 1) << (2 * k)) * 8 < n) ++k;
  const int bits = 2 * k + (in.sphere ? 3 : 0) + prob_bits;

  OrderDev a;
  a.seg[0] = Segment{in.tx, in.ty, in.tz, nullptr, in.i0, in.nt};
  a.seg[1] = Segment{in.x, in.y, in.z, in.list, 0, in.ns};
  a.k = k;
  a.sphere = in.sphere ? 1 : 0;
  a.box = box;
  a.prob = in.prob;
  a.sorted = in.sorted;
  if (!in.sphere) hipLaunchKernelGGL(box_partial, dim3(kBoxBlocks), dim3(256), 0, ctx->stream, a, box);
  hipLaunchKernelGGL(make_keys, dim3((items + 255) / 256), dim3(256), 0, ctx->stream, a, w.key[0], w.val[0]);
  sort_pairs(ctx->stream, w, in.nt, in.ns, bits, tout, sout);
  LPM_HIP(ctx, hipGetLastError());
  return LPM_OK;
}

}  // namespace lpm
