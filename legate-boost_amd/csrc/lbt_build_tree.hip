// BuildTreeTask for one MI355X: split-proposal gather, gradient quantisation,
// per-level histograms (LDS-privatised, merged by 64-bit integer atomics),
// prefix scan + sibling subtraction, split evaluation with the reference's
// tie rule, and the stable row->node partition.
//
// Semantics follow rapidsai/legate-boost src/models/tree/build_tree.cu and
// build_tree.h (cited per kernel); the decomposition into kernels is this
// library's own and is written for gfx950 (64-wide waves, 160 KB LDS per CU).
#include "lbt_device.h"
#include "lbt_internal.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <type_traits>

namespace lbt {
namespace {

constexpr int kThreads = 256;

// ---------------------------------------------------------------------------
// tree initialisation / output (build_tree.cu:785-861)
// ---------------------------------------------------------------------------

// Also what the TreeBuilder's constructor sets up (build_tree.cu:967-974, every row starts in the
// root) and the per-level counters.
struct InitArgs {
  double* leaf;
  int32_t* feature;
  double* split;
  double* gain;
  I64Pair* node_sums;
  int64_t max_nodes;
  int K;
  int32_t* rows;
  int64_t n;
  int32_t* seg;
  int32_t* block_seg;
  int64_t n_slabs;
  uint4* level_totals;
  int n_totals16;
  uint8_t* tainted;
  __device__ __forceinline__ void entry(int64_t i) const
  {
    if (i < max_nodes * K) {
      leaf[i]      = 0.0;
      node_sums[i] = I64Pair{0, 0};
    }
    if (i < max_nodes) {
      feature[i] = -1;
      split[i]   = 0.0;
      gain[i]    = 0.0;
      tainted[i] = 0;
    }
    if (i < n) rows[i] = static_cast<int32_t>(i);
    if (i < n_slabs) block_seg[i] = 0;
    if (i < n_totals16) level_totals[i] = make_uint4(0, 0, 0, 0);
    if (i == 0) {
      seg[0] = 0;
      seg[1] = static_cast<int32_t>(n);
    }
  }
};

__global__ void write_hessian_kernel(double* hessian, const I64Pair* node_sums, int64_t n,
                                     const double* scales)
{
  int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (i < n) hessian[i] = static_cast<double>(node_sums[i].hess) * scales[3];
}

__global__ void zero_kernel(uint4* p, int64_t n16)
{
  int64_t i      = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (; i < n16; i += stride) p[i] = make_uint4(0, 0, 0, 0);
}

// Clears the node's histogram if rows will be added to it: of two siblings one, the other one is written whole by the scan. `parts`
// workgroups share a node.
__device__ __forceinline__ void clear_built(const HistView& hist, const I64Pair* node_sums, int node, int part, int parts)
{
  if (node_sums[static_cast<int64_t>(node) * hist.K].hess <= 0) return;
  if (!hist.builds(node, node_sums)) return;
  uint4* const p   = reinterpret_cast<uint4*>(hist.at(node, 0, 0));
  const int64_t n  = static_cast<int64_t>(hist.K) * hist.B;
  const int64_t st = static_cast<int64_t>(parts) * kThreads;
  for (int64_t i = part * static_cast<int64_t>(kThreads) + threadIdx.x; i < n; i += st) p[i] = make_uint4(0, 0, 0, 0);
}
__global__ void __launch_bounds__(kThreads) zero_built_kernel(HistView hist, const I64Pair* node_sums, int node_begin)
{
  clear_built(hist, node_sums, node_begin + blockIdx.x, blockIdx.y, gridDim.y);
}

// ---------------------------------------------------------------------------
// split proposals (build_tree.cu:867-964)
// ---------------------------------------------------------------------------

template <typename T>
struct SampleArgs {
  const T* X;
  int64_t row_offset, n_rows, dataset_rows;
  int F, S, P;  // features, samples, the power of two that holds them
  int32_t seed;
  T* uniq;          // [F][S]
  int32_t* counts;  // [F]
  int32_t* row_pointers;
  T* proposals;
  int32_t* bin_feature;
  double* as_double;           // optional: the proposals as doubles, what WriteTreeOutput stores as split values
  int32_t* host_row_pointers;  // optional: the row pointers for the host, F + 1 words
};

// Sum over a workgroup of 256, and what lies in front of the thread.
__device__ __forceinline__ int sum_before(int mine, int* s_waves, int* all)
{
  const int incl = static_cast<int>(wave_inclusive_sum32(static_cast<uint32_t>(mine)));
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 63) s_waves[wave] = incl;
  __syncthreads();
  int before = incl - mine, total = 0;
  for (int w = 0; w < kThreads / 64; w++) {
    before += w < wave ? s_waves[w] : 0;
    total += s_waves[w];
  }
  *all = total;
  return before;
}

// A workgroup's feature: the S sampled rows' values, row_i from a fresh minstd engine advanced by i (build_tree.cu:882-898),
// sorted in the LDS on order-preserving integer keys, without those equal to their predecessor (thrust::sort +
// unique_copy, build_tree.cu:908-931).
template <typename T>
__device__ __forceinline__ void unique_samples(const SampleArgs<T>& a, int f, typename KeyOf<T>::type* keys, int* s_waves)
{
  using Key = typename KeyOf<T>::type;
  for (int i = threadIdx.x; i < a.P; i += kThreads) {
    Key key = ~Key(0);
    if (i < a.S) {
      const uint32_t x = minstd_next(minstd_discard(minstd_seed(static_cast<uint32_t>(a.seed)), static_cast<uint64_t>(i)));
      const double u   = uniform01(x);
      const double b   = static_cast<double>(a.dataset_rows - 1) + 1.0;
      const int64_t row = static_cast<int64_t>((u * (b - 0.0)) + 0.0);
      const bool has    = row >= a.row_offset && row <= a.row_offset + a.n_rows - 1;
      key = to_key(has ? a.X[(row - a.row_offset) * a.F + f] : T(0));
    }
    keys[i] = key;
  }
  __syncthreads();
  for (int size = 2; size <= a.P; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = threadIdx.x; i < a.P / 2; i += kThreads) {
        int lo      = 2 * i - (i & (stride - 1));  // index with the stride bit clear
        int hi      = lo + stride;
        bool up     = (lo & size) == 0;
        Key x = keys[lo], y = keys[hi];
        if ((x > y) == up) {
          keys[lo] = y;
          keys[hi] = x;
        }
      }
      __syncthreads();
    }
  }
  // thread t owns the contiguous slice [t*per, (t+1)*per)
  const int per = (a.S + kThreads - 1) / kThreads;
  const int begin = min(a.S, static_cast<int>(threadIdx.x) * per), end = min(a.S, begin + per);
  int cnt = 0;
  for (int i = begin; i < end; i++) {
    bool keep = i == 0 || !(from_key(keys[i]) == from_key(keys[i - 1]));
    cnt += keep ? 1 : 0;
  }
  int all = 0;
  int at  = sum_before(cnt, s_waves, &all);
  if (threadIdx.x == 0) a.counts[f] = all;
  T* dst = a.uniq + static_cast<int64_t>(f) * a.S;
  for (int i = begin; i < end; i++) {
    bool keep = i == 0 || !(from_key(keys[i]) == from_key(keys[i - 1]));
    if (keep) dst[at++] = from_key(keys[i]);
  }
}

// What the host waits for a kernel stores in the pinned words of host_mirror: a copy behind the kernel takes 4 us on the
// device and leaves 5 more in front of the next launch (two of them; a fit of 1,000,000 x 50, 4 rounds of depth 12: 6.37 ms
// with, 6.27 without). Wide inputs are copied: one workgroup's words over PCIe would take longer.
constexpr int kMirrorFeatures = 4096;
__device__ __forceinline__ void store_for_host(int32_t* to, int32_t v)
{
  __hip_atomic_store(to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A workgroup's run of features: their CSR row pointers (reduce_by_key + inclusive_scan, build_tree.cu:933-949) and their proposals in
// their place, the last one of each +inf (build_tree.cu:953-956). What lies in front of the run every workgroup adds up for itself, from the
// counts of the launch before. There are no more than kPlaceGroups workgroups, else these loads grow with the square of the features: both
// launches of the proposals with 2 samples of 100,000 and 262,144 features 1118 and 6971 us by a workgroup a feature; by 512 runs 147 and 364, 1024
// 124 and 306, 2048 113 and 280, 4096 122 and 302. (As four launches with one workgroup's scan of the counts 450 and 1053.) Up to 2048
// features a run is one: 500 with 256 samples 13.8 us.
constexpr int kPlaceGroups = 2048;
template <typename T>
__device__ __forceinline__ void place_proposals(const SampleArgs<T>& a, int f0, int f1, int* s_waves)
{
  int mine = 0, b0 = 0;
#pragma unroll 8
  for (int i = threadIdx.x; i < f0; i += kThreads) mine += a.counts[i];
  sum_before(mine, s_waves, &b0);
  for (int f = f0; f < f1; f++) {
    const int n = a.counts[f];
    if (threadIdx.x == 0) {
      a.row_pointers[f + 1] = b0 + n;
      if (f == 0) a.row_pointers[0] = 0;
      if (a.host_row_pointers != nullptr) {
        store_for_host(a.host_row_pointers + f + 1, b0 + n);
        if (f == 0) store_for_host(a.host_row_pointers, 0);
      }
    }
    for (int i = threadIdx.x; i < n; i += kThreads) {
      T v = a.uniq[static_cast<int64_t>(f) * a.S + i];
      if (i == n - 1) v = std::numeric_limits<T>::infinity();
      a.proposals[b0 + i]   = v;
      a.bin_feature[b0 + i] = f;
      if (a.as_double != nullptr) a.as_double[b0 + i] = static_cast<double>(v);
    }
    b0 += n;
  }
}

// ---------------------------------------------------------------------------
// gradient quantiser (build_tree.cu:51-140, :168-204)
// ---------------------------------------------------------------------------

// One level of the fixed-order sum: chunk c covers 4096 entries; lane t adds
// entries t, t+256, ... in order, then a binary tree (strides 128..1) joins the
// 256 lanes. The reference leaves this order to thrust::reduce
// (build_tree.cu:82-83); fixing it makes the two scale factors reproducible.
constexpr int kSumChunk = 4096;
struct TwoSums {
  double a[kThreads], b[kThreads];
};
template <bool kAbs>
__device__ __forceinline__ void sum_chunk(const double* a, const double* b, int64_t n, int64_t c, TwoSums& s)
{
  double xa = 0.0, xb = 0.0;
  for (int j = 0; j < kSumChunk / kThreads; j++) {
    int64_t e = c * kSumChunk + threadIdx.x + static_cast<int64_t>(kThreads) * j;
    if (e < n) {
      xa += kAbs ? fabs(a[e]) : a[e];
      xb += kAbs ? fabs(b[e]) : b[e];
    }
  }
  s.a[threadIdx.x] = xa;
  s.b[threadIdx.x] = xb;
  __syncthreads();
  for (int stride = kThreads / 2; stride >= 1; stride >>= 1) {
    if (static_cast<int>(threadIdx.x) < stride) {
      s.a[threadIdx.x] += s.a[threadIdx.x + stride];
      s.b[threadIdx.x] += s.b[threadIdx.x + stride];
    }
    __syncthreads();
  }
}
__global__ void __launch_bounds__(kThreads)
  sum_level_kernel(const double* a, const double* b, int64_t n, double* out_a, double* out_b)
{
  __shared__ TwoSums s;
  sum_chunk<false>(a, b, n, blockIdx.x, s);
  if (threadIdx.x == 0) {
    out_a[blockIdx.x] = s.a[0];
    out_b[blockIdx.x] = s.b[0];
  }
}

// qstats[0] = max over all entries of max(|q.grad|, |q.hess|); qstats[1]: bits of what was met.
constexpr unsigned kQuantTooLarge        = 1u;  // a value does not fit the packed int32 form (|q| = 2^31: a single
                                                // entry that holds the whole absolute sum, rounded up)
constexpr unsigned kQuantHessNotPositive = 2u;  // an entry that is not (0, 0) and whose hessian is not positive
constexpr unsigned kQuantHessNegative    = 4u;  // an entry whose hessian is negative

// The absolute sums of the gradients up to one that one workgroup adds, and the scales.
struct SumArgs {
  const double* g;
  const double* h;
  int64_t n;
  int m;                // chunks of g and h to add; 0: the caller has their sums
  double* first[2];     // [chunks] their sums
  const double* of[2];  // what the last level adds,
  int n_of;             // so many
  double* scales;       // null: no sums are wanted
  unsigned long long* qstats;
};
__device__ __forceinline__ void find_scales(const SumArgs& a, TwoSums& s)
{
  double sum_a, sum_b;
  if (a.n_of > 1) {
    sum_chunk<false>(a.of[0], a.of[1], a.n_of, 0, s);
    sum_a = s.a[0], sum_b = s.b[0];
  } else {
    sum_a = a.of[0][0], sum_b = a.of[1][0];
  }
  if (threadIdx.x == 0) {
    const double max_int = 2147483647.0;
    double sg = sum_a == 0 ? 1 : max_int / sum_a;
    double sh = sum_b == 0 ? 1 : max_int / sum_b;
    a.scales[0] = sg;
    a.scales[1] = sh;
    a.scales[2] = 1.0 / sg;
    a.scales[3] = 1.0 / sh;
    a.qstats[0] = 0;
    a.qstats[1] = 0;
  }
}

// A tree begins in two launches of workgroups that do one thing each. The first: the features' sorted samples, the first level of
// the absolute sums, and n_init workgroups of the state. The second: the proposals' places, and (one more workgroup, where they are
// wanted) the sums' last level and the scales. Apart they were eight launches, each a chain of few loads, up to the
// rounding of the gradients 58 us of a tree of 1,000,000 x 50, now 27 (of the sort's 13 us 7 were one thread's sum of 256 counts).
template <typename T>
__global__ void __launch_bounds__(kThreads) tree_start_kernel(SampleArgs<T> a, SumArgs sums, InitArgs init)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ TwoSums s_sums;
  __shared__ int s_waves[kThreads / 64];
  int id = static_cast<int>(blockIdx.x);
  // neighbouring features, whose samples share cache lines, on one XCD
  const int per = (a.F + 7) / 8;
  if (id < 8 * per) {
    const int f = (id & 7) * per + (id >> 3);
    if (f < a.F) unique_samples(a, f, reinterpret_cast<typename KeyOf<T>::type*>(smem_raw), s_waves);
    return;
  }
  id -= 8 * per;
  if (id < sums.m) {
    sum_chunk<true>(sums.g, sums.h, sums.n, id, s_sums);
    if (threadIdx.x == 0) {
      sums.first[0][id] = s_sums.a[0];
      sums.first[1][id] = s_sums.b[0];
    }
    return;
  }
  init.entry(static_cast<int64_t>(id - sums.m) * kThreads + threadIdx.x);
}
template <typename T>
__global__ void __launch_bounds__(kThreads) tree_scales_kernel(SampleArgs<T> a, int run, SumArgs sums)
{
  __shared__ TwoSums s_sums;
  __shared__ int s_waves[kThreads / 64];
  const int f = static_cast<int>(blockIdx.x) * run;  // (in range: no more than kPlaceGroups + 1 workgroups of ceil(F / kPlaceGroups))
  if (f < a.F)
    place_proposals(a, f, min(a.F, f + run), s_waves);
  else
    find_scales(sums, s_sums);
}

// Stochastic rounding of every (row, output) once per tree, stored as int32
// pairs, plus the root sums (build_tree.cu:112-129, :168-204). The reference
// redoes this rounding inside every histogram launch; the values are the same.
// Bound by memory for many rows. For fewer it is the workgroups' three additions to the same words, which take turns
// of about 9 ns: 2048 workgroups of 256 threads took 53 us for 1,000,000 rows, 256 of 1024 take 14 (10,000,000
// rows: 67, now 53). A thread asks for the rows of its next kQuantiseRows turns together.
constexpr int kQuantiseThreads = 1024, kQuantiseGroups = 256, kQuantiseRows = 4;
__global__ void __launch_bounds__(kQuantiseThreads)
  quantise_kernel(const double* g, const double* h, int64_t n_rows, int K, int64_t row_offset,
                  int64_t seed, const double* scales, int2* q_out, I64Pair* node_sums,
                  unsigned long long* qstats)
{
  __shared__ int64_t s_g[kQuantiseThreads / 64];
  __shared__ int64_t s_h[kQuantiseThreads / 64];
  __shared__ unsigned long long s_m[kQuantiseThreads / 64];
  __shared__ unsigned s_bad[kQuantiseThreads / 64];
  const int k = blockIdx.y;
  const double sg = scales[0], sh = scales[1];
  int64_t sum_g = 0, sum_h = 0;
  unsigned long long mx = 0;
  unsigned bad = 0;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kQuantiseThreads;
  auto round_row = [&](int64_t row, double grad, double hess) {
    int64_t qg, qh;
    quantise_pair(grad, hess, sg, sh, seed, row + row_offset, static_cast<int64_t>(k), &qg, &qh);
    bad |= qg > 2147483647LL || qg < -2147483647LL || qh > 2147483647LL || qh < -2147483647LL ? kQuantTooLarge : 0;
    bad |= qh <= 0 && (qg != 0 || qh != 0) ? kQuantHessNotPositive : 0;
    bad |= qh < 0 ? kQuantHessNegative : 0;
    q_out[row * K + k] = make_int2(static_cast<int>(qg), static_cast<int>(qh));
    unsigned long long ag = static_cast<unsigned long long>(qg < 0 ? -qg : qg);
    unsigned long long ah = static_cast<unsigned long long>(qh < 0 ? -qh : qh);
    mx = ag > mx ? ag : mx;
    mx = ah > mx ? ah : mx;
    sum_g += qg;
    sum_h += qh;
  };
  for (int64_t row = blockIdx.x * static_cast<int64_t>(kQuantiseThreads) + threadIdx.x; row < n_rows;
       row += kQuantiseRows * stride) {
    double grad[kQuantiseRows], hess[kQuantiseRows];
#pragma unroll
    for (int u = 0; u < kQuantiseRows; u++) {
      const int64_t at = row + u * stride < n_rows ? row + u * stride : row;
      grad[u] = g[at * K + k];
      hess[u] = h[at * K + k];
    }
#pragma unroll
    for (int u = 0; u < kQuantiseRows; u++)
      if (row + u * stride < n_rows) round_row(row + u * stride, grad[u], hess[u]);
  }
  for (int off = 32; off >= 1; off >>= 1) {
    sum_g += __shfl_down(sum_g, off, 64);
    sum_h += __shfl_down(sum_h, off, 64);
    unsigned long long o = __shfl_down(mx, off, 64);
    mx = o > mx ? o : mx;
    bad |= __shfl_down(bad, off, 64);
  }
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  if (lane == 0) {
    s_g[wave] = sum_g;
    s_h[wave] = sum_h;
    s_m[wave] = mx;
    s_bad[wave] = bad;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kQuantiseThreads / 64; w++) {
      sum_g += s_g[w];
      sum_h += s_h[w];
      mx = s_m[w] > mx ? s_m[w] : mx;
      bad |= s_bad[w];
    }
    atomic_add_i64(&node_sums[k].grad, sum_g);
    atomic_add_i64(&node_sums[k].hess, sum_h);
    atomicMax(&qstats[0], mx);
    if (bad != 0) atomicOr(&qstats[1], static_cast<unsigned long long>(bad));
  }
}

// The same for several outputs per row: the (row, output) entries are walked in memory order
// (the kernel above, launched once per output, would read every line K times). The grid stride
// is a multiple of K, so a thread stays with one output and sums in registers; the outputs'
// sums of a workgroup meet in LDS. As above few workgroups, whose additions to the same 2 K words take turns, and loads of the next turns
// together: 300,000 rows of 16 outputs 102 -> 37 us, 2,000,000 of 8 110 -> 98.
constexpr int kQuantiseFlatMaxK = 2048;
__global__ void __launch_bounds__(kQuantiseThreads)
  quantise_flat_kernel(const double* g, const double* h, int64_t n_rows, int K, int64_t row_offset, int64_t seed,
                       const double* scales, int2* q_out, I64Pair* node_sums, unsigned long long* qstats)
{
  extern __shared__ unsigned long long s_sums[];  // [K] grad, [K] hess
  __shared__ unsigned long long s_max;
  __shared__ unsigned s_bad;
  for (int i = threadIdx.x; i < 2 * K; i += kQuantiseThreads) s_sums[i] = 0;
  if (threadIdx.x == 0) s_max = s_bad = 0;
  __syncthreads();
  const double sg = scales[0], sh = scales[1];
  const int64_t n       = n_rows * K;
  const int64_t threads = static_cast<int64_t>(gridDim.x) * kQuantiseThreads;
  const int64_t stride  = threads / K * K;  // the launch makes sure that threads >= K
  const int64_t first   = blockIdx.x * static_cast<int64_t>(kQuantiseThreads) + threadIdx.x;
  const int k           = static_cast<int>(first % K);
  int64_t sum_g = 0, sum_h = 0;
  unsigned long long mx = 0;
  unsigned bad = 0;
  if (first < stride) {
    auto round_entry = [&](int64_t e, int64_t row, double grad, double hess) {
      int64_t qg, qh;
      quantise_pair(grad, hess, sg, sh, seed, row + row_offset, static_cast<int64_t>(k), &qg, &qh);
      bad |= qg > 2147483647LL || qg < -2147483647LL || qh > 2147483647LL || qh < -2147483647LL ? kQuantTooLarge : 0;
      bad |= qh <= 0 && (qg != 0 || qh != 0) ? kQuantHessNotPositive : 0;
      bad |= qh < 0 ? kQuantHessNegative : 0;
      q_out[e] = make_int2(static_cast<int>(qg), static_cast<int>(qh));
      unsigned long long ag = static_cast<unsigned long long>(qg < 0 ? -qg : qg);
      unsigned long long ah = static_cast<unsigned long long>(qh < 0 ? -qh : qh);
      mx = ag > mx ? ag : mx;
      mx = ah > mx ? ah : mx;
      sum_g += qg;
      sum_h += qh;
    };
    const int64_t step = stride / K;  // rows that a turn moves on
    int64_t row        = first / K;
    for (int64_t e = first; e < n; e += kQuantiseRows * stride, row += kQuantiseRows * step) {
      double grad[kQuantiseRows], hess[kQuantiseRows];
#pragma unroll
      for (int u = 0; u < kQuantiseRows; u++) {
        const int64_t at = e + u * stride < n ? e + u * stride : e;
        grad[u] = g[at];
        hess[u] = h[at];
      }
#pragma unroll
      for (int u = 0; u < kQuantiseRows; u++)
        if (e + u * stride < n) round_entry(e + u * stride, row + u * step, grad[u], hess[u]);
    }
    atomicAdd(&s_sums[k], static_cast<unsigned long long>(sum_g));
    atomicAdd(&s_sums[K + k], static_cast<unsigned long long>(sum_h));
    atomicMax(&s_max, mx);
  }
  if (bad != 0) atomicOr(&s_bad, bad);
  __syncthreads();
  for (int i = threadIdx.x; i < K; i += kQuantiseThreads) {
    const unsigned long long vg = s_sums[i], vh = s_sums[K + i];
    if (vg != 0) atomic_add_i64(&node_sums[i].grad, static_cast<int64_t>(vg));
    if (vh != 0) atomic_add_i64(&node_sums[i].hess, static_cast<int64_t>(vh));
  }
  if (threadIdx.x == 0) {
    atomicMax(&qstats[0], s_max);
    if (s_bad != 0) atomicOr(&qstats[1], static_cast<unsigned long long>(s_bad));
  }
}

// ---------------------------------------------------------------------------
// scan + sibling subtraction (build_tree.cu:597-668), one wave per
// (feature, node), 64 bins per step
// ---------------------------------------------------------------------------

// taint: where the nodes are told of whose derived histogram is not what their rows add up to (see build_tree_impl); null: nobody asks
__global__ void __launch_bounds__(kThreads)
  scan_kernel(HistView hist, const I64Pair* node_sums, int F, const int32_t* row_pointers,
              int node_begin, int n_nodes, uint8_t* taint)
{
  const int lane     = threadIdx.x & 63;
  const int64_t rank = (blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x) >> 6;
  const int i        = static_cast<int>(rank / n_nodes);
  const int j        = static_cast<int>(rank % n_nodes);
  const int k        = blockIdx.y;
  if (i >= F) return;
  const int node   = node_begin + j;
  const int parent = parent_of(node);
  if (node_sums[static_cast<int64_t>(node) * hist.K + k].hess <= 0) return;
  if (!hist.builds(node, node_sums)) return;
  const bool clean = hist.tainted != nullptr;
  bool unscanned   = false;  // a bin that keeps something else than the running sums

  const int fb = row_pointers[i], fe = row_pointers[i + 1];
  int64_t agg_g = 0, agg_h = 0;
  for (int base = fb; base < fe; base += 64) {
    const int bin  = base + lane;
    const bool in  = bin < fe;
    I64Pair* cell  = hist.at(node, k, in ? bin : fb);
    int64_t eg = wave_inclusive_sum(in ? cell->grad : 0), eh = wave_inclusive_sum(in ? cell->hess : 0);
    int64_t tile_g = wave_read_lane(eg, 63), tile_h = wave_read_lane(eh, 63);
    eg += agg_g;
    eh += agg_h;
    // the reference skips the store when the running sum is not positive
    // (build_tree.cu:645); the raw bin value then stays in place
    if (in && (clean || eg > 0 || eh > 0)) {
      cell->grad = eg;
      cell->hess = eh;
    } else if (in) {
      unscanned |= cell->grad != eg || cell->hess != eh;
    }
    agg_g += tile_g;
    agg_h += tile_h;
  }
  if (node == 0) return;
  const int sib = sibling_of(node);
  if (!hist.builds(sib, node_sums)) {
    if (taint != nullptr && (__any(unscanned) || taint[parent] != 0) && lane == 0) taint[sib] = 1;
    for (int bin = fb + lane; bin < fe; bin += 64) {
      I64Pair s = *hist.at(node, k, bin);
      I64Pair p = *hist.at(parent, k, bin);
      *hist.at(sib, k, bin) = I64Pair{p.grad - s.grad, p.hess - s.hess};
    }
  }
}

// ---------------------------------------------------------------------------
// split evaluation (build_tree.cu:682-782)
// ---------------------------------------------------------------------------

constexpr int kSplitChunk = 2048;  // bins per workgroup

__device__ inline Cand block_best(Cand c, Cand* s_c)
{
  for (int off = 32; off >= 1; off >>= 1) {
    Cand o;
    o.gain = __shfl_down(c.gain, off, 64);
    o.bin  = __shfl_down(c.bin, off, 64);
    if (cand_better(o, c)) c = o;
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) s_c[wave] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < static_cast<int>(blockDim.x) >> 6; w++)
      if (cand_better(s_c[w], c)) c = s_c[w];
  }
  return c;  // valid on thread 0
}

__global__ void __launch_bounds__(kThreads)
  split_eval_kernel(HistView hist, const I64Pair* node_sums, const int32_t* bin_feature,
                    const uint8_t* feature_set, const double* scales, double l1, double l2,
                    double min_split_gain, int node_begin, int n_chunks, Cand* partial)
{
  __shared__ Cand s_c[kThreads / 64];
  const int node = node_begin + blockIdx.x;
  const int K    = hist.K;
  if (node_sums[static_cast<int64_t>(node) * K].hess <= 0) return;
  const double inv_g = scales[2], inv_h = scales[3];
  const double reg   = 1e-5 > l2 ? 1e-5 : l2;
  const int b_lo     = blockIdx.y * kSplitChunk;
  const int b_hi     = min(hist.B, b_lo + kSplitChunk);
  Cand best{0.0, -1};
  for (int bin = b_lo + threadIdx.x; bin < b_hi; bin += kThreads) {
    if (feature_set != nullptr && !feature_set[bin_feature[bin]]) continue;
    double gain = 0;
    for (int k = 0; k < K; k++) {
      I64Pair ns = node_sums[static_cast<int64_t>(node) * K + k];
      I64Pair ls = *hist.at(node, k, bin);
      int64_t rg = ns.grad - ls.grad, rh = ns.hess - ls.hess;
      if (ls.hess <= 0 || rh <= 0) {
        gain = 0;
        break;
      }
      gain += calculate_gain(static_cast<double>(ls.grad) * inv_g, static_cast<double>(ls.hess) * inv_h,
                             static_cast<double>(rg) * inv_g, static_cast<double>(rh) * inv_h,
                             static_cast<double>(ns.grad) * inv_g, static_cast<double>(ns.hess) * inv_h,
                             l1, reg, min_split_gain);
    }
    if (gain > 0) {
      Cand c{gain, bin};
      if (cand_better(c, best)) best = c;
    }
  }
  best = block_best(best, s_c);
  if (threadIdx.x == 0) partial[static_cast<int64_t>(blockIdx.x) * n_chunks + blockIdx.y] = best;
}

// store == false: nothing reads these histograms after the split of their nodes has been applied
// (the last level, or the level before one that starts a new histogram buffer), so the running
// sums and the derived siblings are not written back; split_apply_kernel then forms the one bin
// it needs from the bins as they were accumulated (stored_bin_value).
// Scan, sibling subtraction and split evaluation in one pass over the histograms
// (build_tree.cu:597-668 and :682-740): one wave per (built node, feature) takes 64 bins of the
// feature at a time and, output by output, forms the running sums, stores them under the
// reference's rule, derives the sibling's bins where the sibling is not built, and adds the
// output's share to the gain of every bin of the node and of the sibling while the sums are
// still in registers. The histograms are read once instead of twice, and the candidates of a
// node come out per feature (split_apply_kernel reduces them with the same total order).
// Where the reference's scan returns early for an output (node sum of hessians not positive,
// :613) the bins of that output stay as they are in memory, for the node and for its sibling,
// and the gains are formed from those values, as the reference's split kernel would read them.
//
// Bound by its instructions, and by memory where it stores what it scanned (2,000,000 x 200 with 8 outputs: 64 nodes 0.84 GB read and
// written in 120 us). What a wave shares is told to the compiler (the number of its wave), so that
// addresses and conditions are scalar; the nodes' sums and the gain terms that do not depend on the bin are formed once,
// in lane k for output k (in the loop they were a third of the quotients, and the sibling's sums a load to wait for per
// tile and output); and the four quotients of a bin and its sibling's have no branch between them. Sums are formed in 32 bits
// (narrow_sums_hold) and turned into doubles from there, differences are differences of doubles, and quotients are formed without
// what only the ends of the exponent need (plain_quotients): of 190 instructions a tile and output without a derived sibling 115
// are left. The 18 launches with a wave a pair of three trees of 2,000,000 x 200 with 8 outputs: 1740 -> 1426 us (32 bits alone
// 1591); the 20 of four trees of 1,000,000 x 50 with 512 samples: 464 -> 402.
// kW: waves that share a (node, feature), see scan_split_launch.
constexpr int kFusedMaxK   = 64;  // lane k of the wave keeps the running sums of output k

// The running sums are formed in their lower 32 bits, one instruction a step where 64 bits take four. The absolute values of an output's
// grads (hessians) sum up to less than 2^31 + N + 1024; with the root's sum G of them, sums over any rows lie between -down and
// up, down = (2^31 + N + 1024 - G) / 2 + 1, up with + G, less than 2^32 apart: the lower half of a sum + down is the sum + down. Whole numbers
// of that size are exact as doubles, and so are their differences.
constexpr bool narrow_sums_hold(int64_t n_rows) { return n_rows < (int64_t(1) << 31) - 4096; }

__device__ __forceinline__ Cand wave_best(const Cand& c)  // the same in every lane
{
  const int from = wave_best_lane(c.gain, c.bin);
  return from < 0 ? Cand{0.0, -1} : Cand{wave_read_lane_f64(c.gain, from), __builtin_amdgcn_readlane(c.bin, from)};
}

template <int kW>
__global__ void __launch_bounds__(kW == 1 ? kThreads : kW * 64)
  scan_split_kernel(HistView hist, const I64Pair* __restrict__ node_sums, int F, const int32_t* __restrict__ row_pointers,
                    int node_begin, int n_nodes, const uint8_t* __restrict__ feature_set,
                    const double* __restrict__ scales, double l1, double l2, double min_split_gain, Cand* partial,
                    int64_t n_rows, bool store, uint8_t* taint)
{
  __shared__ uint2 s_total[kW][kFusedMaxK];
  __shared__ Cand s_best[2][kW];
  const int lane  = threadIdx.x & 63;
  const int wave  = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int slice = kW == 1 ? 0 : wave;  // this wave's share of the feature's tiles
  const int64_t rank = kW == 1 ? static_cast<int64_t>(blockIdx.x) * (kThreads / 64) + wave : blockIdx.x;
  const int i        = static_cast<int>(rank / n_nodes);
  const int j        = static_cast<int>(rank % n_nodes);
  if (i >= F) return;
  const int K      = hist.K;
  const int node   = node_begin + j;
  const int parent = parent_of(node);
  if (!hist.builds(node, node_sums)) return;
  const int sib     = node == 0 ? -1 : sibling_of(node);
  const bool derive = node != 0 && !hist.builds(sib, node_sums);
  const bool clean  = hist.tainted != nullptr;
  bool unscanned    = false;  // a bin that keeps something else than the running sums
  // lane k holds the node's and its sibling's sums of output k and the terms of the gains that do not depend on the bin
  I64Pair sum_n{0, 0}, sum_s{0, 0};
  if (lane < K) {
    sum_n = node_sums[static_cast<int64_t>(node) * K + lane];
    if (derive) sum_s = node_sums[static_cast<int64_t>(sib) * K + lane];
  }
  // which of the two are split candidates at all (build_tree.cu:712), and on this feature
  const bool usable = feature_set == nullptr || feature_set[i] != 0;
  const bool eval_n = usable && wave_read_lane(sum_n.hess, 0) > 0;
  const bool eval_s = usable && derive && wave_read_lane(sum_s.hess, 0) > 0;
  // Nothing to scan (no output of the node has a positive sum of hessians: an empty node, as
  // most nodes of a deep level are) and nothing to evaluate: the bins stay as they are.
  const unsigned long long scans = __ballot(sum_n.hess > 0);
  if (scans == 0 && !eval_n && !eval_s) {
    if (lane == 0 && slice == 0) {
      partial[static_cast<int64_t>(j) * F + i] = Cand{0.0, -1};
      if (derive) partial[static_cast<int64_t>(sib - node_begin) * F + i] = Cand{0.0, -1};
    }
    return;
  }
  const double inv_g = scales[2], inv_h = scales[3];
  const double reg   = 1e-5 > l2 ? 1e-5 : l2;
  const double own_n = leaf_gain(static_cast<double>(sum_n.grad) * inv_g, static_cast<double>(sum_n.hess) * inv_h, l1, reg);
  const double own_s = leaf_gain(static_cast<double>(sum_s.grad) * inv_g, static_cast<double>(sum_s.hess) * inv_h, l1, reg);
  // lane k: the lower halves' origin of output k, see narrow_sums_hold
  uint32_t down_g = 0, down_h = 0;
  if (lane < K) {
    const I64Pair root = node_sums[lane];
    const int64_t most = (int64_t(1) << 31) + n_rows + 1024;
    down_g = static_cast<uint32_t>((most - root.grad) / 2 + 1);
    down_h = static_cast<uint32_t>((most - root.hess) / 2 + 1);
  }
  const double all_ng = static_cast<double>(sum_n.grad), all_nh = static_cast<double>(sum_n.hess);
  const double all_sg = static_cast<double>(sum_s.grad), all_sh = static_cast<double>(sum_s.hess);
  const int fb = row_pointers[i], fe = row_pointers[i + 1];
  const int n_tiles = (fe - fb + 63) / 64;
  const int t0 = n_tiles * slice / kW, t1 = n_tiles * (slice + 1) / kW;
  const I64Pair* const bins_n = hist.at(node, 0, 0);
  const I64Pair* const bins_p = derive ? hist.at(parent, 0, 0) : bins_n;
  const I64Pair* const bins_s = derive ? hist.at(sib, 0, 0) : bins_n;
  uint32_t agg_g = 0, agg_h = 0;  // lane k: sums of output k over the tiles done so far, lower halves
  if constexpr (kW > 1) {
    // every wave adds up its tiles, then takes over the sums of the tiles in front of them
    for (int k = 0; k < K; k++) {
      uint32_t g = 0, h = 0;
      for (int tile = t0; tile < t1; tile++) {
        const int b     = fb + tile * 64 + lane;
        const I64Pair v = bins_n[static_cast<int64_t>(k) * hist.B + min(b, fe - 1)];
        g += b < fe ? static_cast<uint32_t>(v.grad) : 0u;
        h += b < fe ? static_cast<uint32_t>(v.hess) : 0u;
      }
      const uint32_t all_g = wave_inclusive_sum32(g), all_h = wave_inclusive_sum32(h);
      if (lane == 63) s_total[wave][k] = make_uint2(all_g, all_h);
    }
    __syncthreads();
    if (lane < K) {
      for (int w = 0; w < wave; w++) {
        agg_g += s_total[w][lane].x;
        agg_h += s_total[w][lane].y;
      }
    }
  }
  Cand best_n{0.0, -1}, best_s{0.0, -1};
  // The bins of the next (tile, output) and the parent's are requested before the current ones
  // are scanned and stored: the stores would otherwise keep every load behind them, and a wave
  // would wait for memory once per tile and output. (Two or four of them ahead: no faster.)
  const int n_items = (t1 - t0) * K;
  auto run = [&](auto derives, auto plains) {
    constexpr bool kDerive = decltype(derives)::value;
    auto quotient = [&](double grad, double hess) {
      if constexpr (decltype(plains)::value)
        return quotient_plain(grad * grad, hess + reg);
      else
        return leaf_gain_select(grad, hess, l1, reg);
    };
    I64Pair val_next{0, 0}, other_next{0, 0};
    int fetch_t = t0, fetch_k = 0;
    auto fetch = [&]() {
      const int64_t at = static_cast<int64_t>(fetch_k) * hist.B + min(fb + fetch_t * 64 + lane, fe - 1);
      val_next         = bins_n[at];  // what the split evaluation reads for this bin
      // the parent's bin where the sibling is derived from it, else the sibling's bin as it is in memory
      if constexpr (kDerive) other_next = (scans >> fetch_k & 1) != 0 ? bins_p[at] : bins_s[at];
      if (++fetch_k == K) {
        fetch_k = 0;
        fetch_t++;
      }
    };
    if (n_items > 0) fetch();
    int k = 0, bin = fb + t0 * 64 + lane;
    double gain_n = 0.0, gain_s = 0.0;
    bool live_n = true, live_s = true;
    for (int item = 0; item < n_items; item++) {
      const bool in = bin < fe;
      I64Pair val   = in ? val_next : I64Pair{0, 0}, sval = other_next;
      if (item + 1 < n_items) fetch();
      const int64_t at = static_cast<int64_t>(k) * hist.B + bin;
      double lg, lh;  // what lies left of the bin
      if ((scans >> k & 1) != 0) {
        const uint32_t raw_g = static_cast<uint32_t>(val.grad), raw_h = static_cast<uint32_t>(val.hess);
        const uint32_t to_g = wave_inclusive_sum32(raw_g) + wave_read_lane32(agg_g, k);
        const uint32_t to_h = wave_inclusive_sum32(raw_h) + wave_read_lane32(agg_h, k);
        const uint32_t tile_g = wave_read_lane32(to_g, 63), tile_h = wave_read_lane32(to_h, 63);
        if (lane == k) {
          agg_g = tile_g;
          agg_h = tile_h;
        }
        const uint32_t from_g = wave_read_lane32(down_g, k), from_h = wave_read_lane32(down_h, k);
        lg = static_cast<double>(to_g + from_g) - static_cast<double>(from_g);
        lh = static_cast<double>(to_h + from_h) - static_cast<double>(from_h);
        // the reference skips the store when the running sum is not positive
        // (build_tree.cu:645); the raw bin value then stays in place
        const bool positive = clean || lg > 0 || lh > 0;
        if (store) {
          const int64_t eg = static_cast<int64_t>(to_g + from_g) - static_cast<int64_t>(from_g);
          const int64_t eh = static_cast<int64_t>(to_h + from_h) - static_cast<int64_t>(from_h);
          if (in && positive) const_cast<I64Pair*>(bins_n)[at] = I64Pair{eg, eh};
          if constexpr (kDerive) {
            const I64Pair left = positive ? I64Pair{eg, eh} : val;
            if (in) const_cast<I64Pair*>(bins_s)[at] = I64Pair{sval.grad - left.grad, sval.hess - left.hess};
          }
        }
        if (__any(!positive && (to_g | to_h | raw_g | raw_h) != 0)) {  // (else a bin that is not positive is zero, as its sum)
          asm volatile("");  // (a branch: without it both conversions are formed every time)
          unscanned |= in && !positive && (to_g != raw_g || to_h != raw_h);
          lg = positive ? lg : static_cast<double>(val.grad);
          lh = positive ? lh : static_cast<double>(val.hess);
        }
      } else {
        lg = static_cast<double>(val.grad);
        lh = static_cast<double>(val.hess);
      }
      // build_tree.cu:727-730: one output without a valid split on a bin voids the bin. The quotients of
      // the node and of the sibling are formed without branches, so that their chains run side by side. (All sums are whole
      // numbers below 2^35, and so are their differences as doubles.)
      const double rg = wave_read_lane_f64(all_ng, k) - lg, rh = wave_read_lane_f64(all_nh, k) - lh;
      live_n = live_n && lh > 0 && rh > 0;
      const double left_n  = quotient(lg * inv_g, lh * inv_h);
      const double right_n = quotient(rg * inv_g, rh * inv_h);
      double left_s = 0.0, right_s = 0.0;
      if constexpr (kDerive) {
        const bool derived = (scans >> k & 1) != 0;
        const double slg = static_cast<double>(sval.grad) - (derived ? lg : 0.0), slh = static_cast<double>(sval.hess) - (derived ? lh : 0.0);
        const double srg = wave_read_lane_f64(all_sg, k) - slg, srh = wave_read_lane_f64(all_sh, k) - slh;
        live_s  = live_s && slh > 0 && srh > 0;
        left_s  = quotient(slg * inv_g, slh * inv_h);
        right_s = quotient(srg * inv_g, srh * inv_h);
      }
      gain_n += 0.5 * (left_n + right_n - wave_read_lane_f64(own_n, k)) - min_split_gain;
      if constexpr (kDerive) gain_s += 0.5 * (left_s + right_s - wave_read_lane_f64(own_s, k)) - min_split_gain;
      if (++k == K) {
        if (in && eval_n && live_n && gain_n > 0) {
          const Cand c{gain_n, bin};
          if (cand_better(c, best_n)) best_n = c;
        }
        if (kDerive && in && eval_s && live_s && gain_s > 0) {
          const Cand c{gain_s, bin};
          if (cand_better(c, best_s)) best_s = c;
        }
        k = 0;
        bin += 64;
        gain_n = gain_s = 0.0;
        live_n = live_s = true;
      }
    }
  };
  if (plain_quotients(l1, inv_g, inv_h, reg)) {
    if (derive)
      run(std::true_type{}, std::true_type{});
    else
      run(std::false_type{}, std::true_type{});
  } else {
    if (derive)
      run(std::true_type{}, std::false_type{});
    else
      run(std::false_type{}, std::false_type{});
  }
  if (derive && taint != nullptr && (__any(unscanned) || taint[parent] != 0) && lane == 0) taint[sib] = 1;
  best_n = wave_best(best_n);
  if (derive) best_s = wave_best(best_s);
  if constexpr (kW > 1) {
    if (lane == 0) {
      s_best[0][wave] = best_n;
      s_best[1][wave] = best_s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < kW; w++) {
        if (cand_better(s_best[0][w], best_n)) best_n = s_best[0][w];
        if (cand_better(s_best[1][w], best_s)) best_s = s_best[1][w];
      }
    }
  }
  if (lane == 0 && slice == 0) {
    partial[static_cast<int64_t>(j) * F + i] = best_n;
    if (derive) partial[static_cast<int64_t>(sib - node_begin) * F + i] = best_s;
  }
}

// Up to 512 (node, feature) pairs a workgroup shares a pair's tiles, a wave each for up to eight of them: such
// levels leave most of the chip idle, and a wave's tiles are a chain (us, eight against one wave, 300,000 x 50 with
// 512 samples: 50 pairs 6.6 : 8.4, 200 8.2 : 12.7, 400 10.9 : 12.0, 800 15.2 : 12.6; four against one with 256: 50 pairs
// 5.5 : 5.9, 400 6.7 : 7.5, 800 9.3 : 7.8). More pairs fill it with one wave each, and the first reading of the shared form,
// for the tiles' sums, is then work on top. A chain is as long as tiles times outputs: with 8 outputs and 512 samples sharing
// pays up to 1280 pairs (64 : 81, 2560 110 : 80), with 3 and 256 up to 400 (11.0 : 14.4, 800 15.3 : 15.4), and with one output
// and two tiles never (50 pairs 5.2 : 4.9, 400 5.8 : 5.0; 3 outputs 400 pairs 8.9 : 9.4, 8 outputs 320 pairs 15.3 : 17.0).
constexpr int64_t kSharedScanPairs = 512;

void scan_split_launch(hipStream_t stream, int max_bins, const HistView& hv, const I64Pair* node_sums, int F,
                       const int32_t* row_pointers, int node_begin, int n_nodes, const uint8_t* feature_set,
                       const double* scales, double l1, double l2, double min_split_gain, Cand* partial, int64_t n_rows, bool store,
                       uint8_t* taint)
{
  const int64_t pairs = static_cast<int64_t>(F) * n_nodes;
  auto launch         = [&](auto kernel, int64_t groups, int threads) {
    kernel<<<static_cast<unsigned>(groups), threads, 0, stream>>>(hv, node_sums, F, row_pointers, node_begin, n_nodes,
                                                                  feature_set, scales, l1, l2, min_split_gain, partial,
                                                                  n_rows, store, taint);
  };
  if (pairs > kSharedScanPairs || max_bins <= (hv.K == 1 ? 128 : 64))
    launch(scan_split_kernel<1>, (pairs + kThreads / 64 - 1) / (kThreads / 64), kThreads);
  else if (max_bins <= 256)
    launch(scan_split_kernel<4>, pairs, 4 * 64);
  else
    launch(scan_split_kernel<8>, pairs, 8 * 64);
}

// What the reference's scan leaves in bin `bin` of (node, output k) of a built node whose bins still
// hold what the rows added: the running sum over the feature's bins up to `bin` where that is
// positive in either half, else the bin as it is (build_tree.cu:645); the bin as it is also where
// the scan returns early for the output (:613). All 64 lanes call this together.
__device__ inline I64Pair stored_bin_value(const HistView& hist, const I64Pair* node_sums, int node, int k, int fb,
                                           int bin, int lane)
{
  const I64Pair raw = *hist.at(node, k, bin);
  if (node_sums[static_cast<int64_t>(node) * hist.K + k].hess <= 0) return raw;
  int64_t g = 0, h = 0;
  for (int b = fb + lane; b <= bin; b += 64) {
    const I64Pair p = *hist.at(node, k, b);
    g += p.grad;
    h += p.hess;
  }
  for (int off = 32; off >= 1; off >>= 1) {
    g += __shfl_xor(g, off, 64);
    h += __shfl_xor(h, off, 64);
  }
  return (hist.tainted != nullptr || g > 0 || h > 0) ? I64Pair{g, h} : raw;
}

// stored == false: scan_split_kernel did not write its results back (see there).
__global__ void __launch_bounds__(64)
  split_apply_kernel(HistView hist, I64Pair* node_sums, const int32_t* bin_feature,
                     const double* proposals_as_double, const double* scales, double l1, double l2,
                     int node_begin, int n_chunks, const Cand* partial, double* leaf,
                     int32_t* feature, double* split, double* gain_out, const int32_t* row_pointers,
                     int32_t* split_bin, bool stored)
{
  __shared__ Cand s_c[1];
  __shared__ Cand s_best;
  const int node = node_begin + blockIdx.x;
  const int K    = hist.K;
  if (node_sums[static_cast<int64_t>(node) * K].hess <= 0) return;
  Cand best{0.0, -1};
  for (int c = threadIdx.x; c < n_chunks; c += 64) {
    Cand o = partial[static_cast<int64_t>(blockIdx.x) * n_chunks + c];
    if (cand_better(o, best)) best = o;
  }
  best = block_best(best, s_c);
  if (threadIdx.x == 0) s_best = best;
  __syncthreads();
  best = s_best;
  if (!(best.bin >= 0 && best.gain > 1e-5)) return;
  const double inv_g = scales[2], inv_h = scales[3];
  const int lc = left_child(node), rc = right_child(node);
  if (!stored) {
    const int lane   = threadIdx.x;
    const int ft     = bin_feature[best.bin];
    const int fb     = row_pointers[ft];
    const int parent = parent_of(node);
    const bool built = hist.builds(node, node_sums);
    for (int k = 0; k < K; k++) {
      const I64Pair ns = node_sums[static_cast<int64_t>(node) * K + k];
      I64Pair ls;
      if (built) {
        ls = stored_bin_value(hist, node_sums, node, k, fb, best.bin, lane);
      } else {
        // derived from its parent and its built sibling, unless the scan of that sibling's output
        // returned early: then the bin is what the buffer holds
        const int sib = sibling_of(node);
        if (node_sums[static_cast<int64_t>(sib) * K + k].hess > 0) {
          const I64Pair sv = stored_bin_value(hist, node_sums, sib, k, fb, best.bin, lane);
          const I64Pair pv = *hist.at(parent, k, best.bin);
          ls               = I64Pair{pv.grad - sv.grad, pv.hess - sv.hess};
        } else {
          ls = *hist.at(node, k, best.bin);
        }
      }
      if (lane == 0) {
        const I64Pair rs{ns.grad - ls.grad, ns.hess - ls.hess};
        node_sums[static_cast<int64_t>(lc) * K + k] = ls;
        node_sums[static_cast<int64_t>(rc) * K + k] = rs;
        leaf[static_cast<int64_t>(lc) * K + k]      = calculate_leaf_value(
          static_cast<double>(ls.grad) * inv_g, static_cast<double>(ls.hess) * inv_h, l1, l2);
        leaf[static_cast<int64_t>(rc) * K + k] = calculate_leaf_value(
          static_cast<double>(rs.grad) * inv_g, static_cast<double>(rs.hess) * inv_h, l1, l2);
        if (k == 0) {
          feature[node]   = ft;
          split[node]     = proposals_as_double[best.bin];
          gain_out[node]  = best.gain;
          split_bin[node] = best.bin - fb;
        }
      }
    }
    return;
  }
  for (int k = threadIdx.x; k < K; k += 64) {
    I64Pair ns = node_sums[static_cast<int64_t>(node) * K + k];
    I64Pair ls = *hist.at(node, k, best.bin);
    I64Pair rs{ns.grad - ls.grad, ns.hess - ls.hess};
    node_sums[static_cast<int64_t>(lc) * K + k] = ls;
    node_sums[static_cast<int64_t>(rc) * K + k] = rs;
    leaf[static_cast<int64_t>(lc) * K + k] = calculate_leaf_value(
      static_cast<double>(ls.grad) * inv_g, static_cast<double>(ls.hess) * inv_h, l1, l2);
    leaf[static_cast<int64_t>(rc) * K + k] = calculate_leaf_value(
      static_cast<double>(rs.grad) * inv_g, static_cast<double>(rs.hess) * inv_h, l1, l2);
    if (k == 0) {
      const int ft    = bin_feature[best.bin];
      feature[node]   = ft;
      split[node]     = proposals_as_double[best.bin];
      gain_out[node]  = best.gain;
      split_bin[node] = best.bin - row_pointers[ft];
    }
  }
}


// ---------------------------------------------------------------------------
// row -> node update and stable partition (build_tree.cu:1026-1080)
// ---------------------------------------------------------------------------
//
// The reference rewrites the node of every (node,row) pair and then runs a
// stable radix sort on the node field. Because the pairs are already sorted by
// node and a node only splits into its two children (or its rows retire with
// key -1), that sort is a stable three-way partition inside every segment:
// retired rows move to the front, then for each parent its left rows followed
// by its right rows. Exclusive prefix counts of the "retired" and "left" flags
// give every destination directly.
//
// The order is held as the list of row numbers alone. The rows of the level's
// node j are the run seg[j] .. seg[j+1] of that list, the rows in front of
// seg[0] have retired, so an index finds its node by its place among the
// segment starts and the node field never travels through memory.

constexpr int kPartItems = 8;
constexpr int kPartBlock = kThreads * kPartItems;  // indices per workgroup ("slab")
constexpr int kSegLds    = kPartBlock + 64;        // segment starts a workgroup keeps in the LDS

// The segments that meet one slab: the one that holds its first index (known per slab,
// block_seg) and the m that start inside it.
struct SlabSegments {
  int j0;       // segment of the slab's first index; -1: it lies among the retired rows
  int m;        // segments j0+1 .. j0+m start inside the slab
  bool in_lds;  // their starts are in the LDS (else they are read from seg)
};

// All threads of the workgroup call this; s_seg has kSegLds entries.
__device__ inline SlabSegments load_slab_segments(const int32_t* __restrict__ seg, int n_parents,
                                                  const int32_t* __restrict__ block_seg, int slab, int64_t base,
                                                  int64_t n, int* s_seg)
{
  SlabSegments ss;
  ss.j0         = block_seg[slab];
  const int end = static_cast<int>(base + kPartBlock < n ? base + kPartBlock : n);
  ss.m          = 0;
  // the starts ascend, so those inside the slab are a prefix of seg[j0+1 ..]
  for (int k = 0;; k += kThreads) {
    const int64_t idx = static_cast<int64_t>(ss.j0) + 1 + k + threadIdx.x;
    const int v       = idx < n_parents ? seg[idx] : 2147483647;
    const bool inside = v < end;
    if (inside && k + static_cast<int>(threadIdx.x) < kSegLds) s_seg[k + threadIdx.x] = v;
    const int cnt = __syncthreads_count(inside);
    ss.m += cnt;
    if (cnt < kThreads) break;
  }
  ss.in_lds = ss.m <= kSegLds;
  return ss;
}

// Segment of index i of the slab (-1: retired): j0 plus the number of starts at or below i.
// Of several segments that start at the same index the last one is not empty.
__device__ inline int segment_of(const SlabSegments& ss, const int* s_seg, const int32_t* __restrict__ seg, int i)
{
  int lo = 0, hi = ss.m;
  if (ss.in_lds) {
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (s_seg[mid] <= i)
        lo = mid + 1;
      else
        hi = mid;
    }
  } else {
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (seg[ss.j0 + 1 + mid] <= i)
        lo = mid + 1;
      else
        hi = mid;
    }
  }
  return ss.j0 + lo;
}

// adds up the per-thread counts of a workgroup and stores them for the scan
__device__ inline void store_block_counts(int nd, int nl, int* s_d, int* s_l, int2* block_counts)
{
  for (int off = 32; off >= 1; off >>= 1) {
    nd += __shfl_down(nd, off, 64);
    nl += __shfl_down(nl, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    s_d[threadIdx.x >> 6] = nd;
    s_l[threadIdx.x >> 6] = nl;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kThreads / 64; w++) {
      nd += s_d[w];
      nl += s_l[w];
    }
    block_counts[blockIdx.x] = make_int2(nd, nl);
  }
}

// pass 1: classify each row (0 retired, 1 left, 2 right) and count per workgroup
template <typename T>
__global__ void __launch_bounds__(kThreads)
  classify_kernel(const int32_t* __restrict__ rows, int64_t n, const int32_t* __restrict__ seg,
                  const int32_t* __restrict__ block_seg, int n_parents, int level_first, const T* X, int F,
                  const int32_t* feature, const double* split, uint8_t* code, int2* block_counts)
{
  __shared__ int s_seg[kSegLds];
  __shared__ int s_d[kThreads / 64];
  __shared__ int s_l[kThreads / 64];
  const int64_t base    = blockIdx.x * static_cast<int64_t>(kPartBlock);
  const SlabSegments ss = load_slab_segments(seg, n_parents, block_seg, blockIdx.x, base, n, s_seg);
  int nd = 0, nl = 0;
#pragma unroll
  for (int u = 0; u < kPartItems; u++) {
    const int64_t i = base + u * kThreads + threadIdx.x;
    if (i < n) {
      const int j = segment_of(ss, s_seg, seg, static_cast<int>(i));
      int c       = 0;
      if (j >= 0) {
        const int node = level_first + j;
        const int ft   = feature[node];
        if (ft != -1) {
          const double xv = static_cast<double>(X[static_cast<int64_t>(rows[i]) * F + ft]);
          c               = xv <= split[node] ? 1 : 2;
        }
      }
      code[i] = static_cast<uint8_t>(c);
      nd += c == 0;
      nl += c == 1;
    }
  }
  store_block_counts(nd, nl, s_d, s_l, block_counts);
}

constexpr int kTransRows = 128;  // the feature-major bins are padded to whole groups of this many rows

// pass 1 when the feature-major bins exist: x <= proposals[b] holds exactly when the
// row's bin (first proposal that is not below x) is <= b, so the split feature's bin
// decides the side and consecutive rows of a node read consecutive bytes.
// kRun: a thread takes eight positions in a row: their row numbers are two loads, their codes one store, and mostly they
// lie in one node; else positions kThreads apart, so that a wave's bins lie close together (see classify_in_runs).
// kDecides: the level's splits have not been applied (split_apply_kernel): every workgroup finds those of the segments that meet its slab, a wave for
// each, and the workgroup in whose slab a segment begins writes the node's outputs: a launch less a level.
struct DecideArgs {
  HistView hist;
  I64Pair* node_sums;
  const int32_t* bin_feature;
  const double* proposals;
  const double* scales;
  double l1, l2;
  int n_cands;  // per node
  const Cand* partial;
  double* leaf;
  int32_t* feature;
  double* split;
  double* gain;
  const int32_t* row_pointers;
  int32_t* split_bin;
};
constexpr int kDecideCands = 512;  // of a node, at most: every slab reads those of its nodes
constexpr int kDecideNodes = 512;
// Every slab reads its nodes' candidates and waits for them, 1 us at 1,000,000 x 50 and 7 at 10,000,000 x 100, whose 4900 slabs are bound by
// what they read; a launch of split_apply_kernel and the gap in front of it are 6 to 7.
constexpr int64_t kDecideRows = int64_t(1) << 22;

// The split of level node j by one wave: feature and bin in every lane, feature -1: none. writes: its outputs as well.
__device__ __forceinline__ int2 decide_node(const DecideArgs& a, int level_first, int j, int lane, bool writes)
{
  const int node = level_first + j, K = a.hist.K;
  const bool usable = a.node_sums[static_cast<int64_t>(node) * K].hess > 0;
  Cand best{0.0, -1};
  for (int c = lane; c < a.n_cands; c += 64) {
    const Cand o = a.partial[static_cast<int64_t>(j) * a.n_cands + c];
    if (cand_better(o, best)) best = o;
  }
  best = wave_best(best);
  if (!usable || !(best.bin >= 0 && best.gain > 1e-5)) return make_int2(-1, 0);
  const int ft = a.bin_feature[best.bin], bin = best.bin - a.row_pointers[ft];
  if (writes) {
    const double inv_g = a.scales[2], inv_h = a.scales[3];
    const int lc = left_child(node), rc = right_child(node);
    if (lane < K) {
      const I64Pair ns = a.node_sums[static_cast<int64_t>(node) * K + lane];
      const I64Pair ls = *a.hist.at(node, lane, best.bin);
      const I64Pair rs{ns.grad - ls.grad, ns.hess - ls.hess};
      a.node_sums[static_cast<int64_t>(lc) * K + lane] = ls;
      a.node_sums[static_cast<int64_t>(rc) * K + lane] = rs;
      a.leaf[static_cast<int64_t>(lc) * K + lane]      = calculate_leaf_value(
        static_cast<double>(ls.grad) * inv_g, static_cast<double>(ls.hess) * inv_h, a.l1, a.l2);
      a.leaf[static_cast<int64_t>(rc) * K + lane] = calculate_leaf_value(
        static_cast<double>(rs.grad) * inv_g, static_cast<double>(rs.hess) * inv_h, a.l1, a.l2);
    }
    if (lane == 0) {
      a.feature[node]   = ft;
      a.split[node]     = a.proposals[best.bin];
      a.gain[node]      = best.gain;
      a.split_bin[node] = bin;
    }
  }
  return make_int2(ft, bin);
}

template <typename BinT, bool kRun, bool kDecides>
__global__ void __launch_bounds__(kThreads)
  classify_bins_kernel(const int32_t* __restrict__ rows, int64_t n, const int32_t* __restrict__ seg,
                       const int32_t* __restrict__ block_seg, int n_parents, int level_first,
                       const BinT* __restrict__ bins_t, int64_t bins_stride, const int32_t* feature,
                       const int32_t* split_bin, uint8_t* code, int2* block_counts, DecideArgs decide)
{
  __shared__ int2 s_split[kDecides ? kDecideNodes + 1 : 1];  // of the slab's segments
  __shared__ int s_seg[kSegLds];
  __shared__ int s_d[kThreads / 64];
  __shared__ int s_l[kThreads / 64];
  const int64_t base = blockIdx.x * static_cast<int64_t>(kPartBlock);
  static_assert(kPartItems == 8, "two 16-byte loads, one 8-byte store");
  const int64_t i0   = base + (kRun ? kPartItems : 1) * static_cast<int64_t>(threadIdx.x);
  constexpr int kGap = kRun ? 1 : kThreads;  // position u of the thread: i0 + u * kGap
  const bool whole   = kRun && i0 + kPartItems <= n;
  // the row numbers are requested before the slab's segments, which they do not depend on
  int row[kPartItems];
  if (whole) {
    const int4 a = *reinterpret_cast<const int4*>(rows + i0), b = *reinterpret_cast<const int4*>(rows + i0 + 4);
    row[0] = a.x, row[1] = a.y, row[2] = a.z, row[3] = a.w;
    row[4] = b.x, row[5] = b.y, row[6] = b.z, row[7] = b.w;
  } else {
#pragma unroll
    for (int u = 0; u < kPartItems; u++) row[u] = i0 + u * kGap < n ? rows[i0 + u * kGap] : 0;
  }
  const SlabSegments ss = load_slab_segments(seg, n_parents, block_seg, blockIdx.x, base, n, s_seg);
  if constexpr (kDecides) {
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    static_assert(kDecideNodes <= kSegLds, "the starts of a level's segments are in the LDS");
    // (an empty segment has no rows that ask, and no split; the others begin in the one slab that has their first position)
    int turn = 0;
    for (int i0 = 0; i0 <= ss.m; i0 += 64) {
      const int i    = i0 + lane;
      const bool has = i <= ss.m && ss.j0 + i >= 0 && (i == ss.m || i == 0 || s_seg[i] > s_seg[i - 1]);
      for (unsigned long long here = __ballot(has); here != 0; here &= here - 1) {
        if ((turn++ & (kThreads / 64 - 1)) != wave) continue;
        const int at    = i0 + __builtin_ctzll(here), j = ss.j0 + at;
        const int begin = at > 0 ? s_seg[at - 1] : seg[j];
        const int2 s    = decide_node(decide, level_first, j, lane, begin >= base);
        if (lane == 0) s_split[at] = s;
      }
    }
    __syncthreads();
  }
  int ft[kPartItems], sb[kPartItems];
  auto look_up = [&](int u, int j) {
    if constexpr (kDecides) {
      const int2 s = j >= 0 ? s_split[j - ss.j0] : make_int2(-1, 0);
      ft[u] = s.x, sb[u] = s.y;
    } else {
      ft[u] = j >= 0 ? feature[level_first + j] : -1;
      sb[u] = j >= 0 ? split_bin[level_first + j] : 0;
    }
  };
  auto segment_at = [&](int64_t i) { return i < n ? segment_of(ss, s_seg, seg, static_cast<int>(i)) : -1; };
  const int first = segment_at(i0);
  look_up(0, first);
#pragma unroll
  for (int u = 1; u < kPartItems; u++) {
    ft[u] = ft[0];
    sb[u] = sb[0];
  }
  if (!whole || first != segment_at(i0 + kPartItems - 1)) {
#pragma unroll
    for (int u = 1; u < kPartItems; u++) look_up(u, segment_at(i0 + u * kGap));
  }
  int bin[kPartItems];
#pragma unroll
  for (int u = 0; u < kPartItems; u++)
    bin[u] = ft[u] != -1 ? static_cast<int>(bins_t[ft[u] * bins_stride + row[u]]) : 0;
  int nd = 0, nl = 0;
  unsigned codes[2] = {0, 0};
#pragma unroll
  for (int u = 0; u < kPartItems; u++) {
    const unsigned c = ft[u] == -1 ? 0u : (bin[u] <= sb[u] ? 1u : 2u);
    const bool here  = i0 + u * kGap < n;
    codes[u >> 2] |= c << (8 * (u & 3));
    if (here && !whole) code[i0 + u * kGap] = static_cast<uint8_t>(c);
    nd += here && c == 0;
    nl += here && c == 1;
  }
  if (whole) *reinterpret_cast<uint2*>(code + i0) = make_uint2(codes[0], codes[1]);
  store_block_counts(nd, nl, s_d, s_l, block_counts);
}

// Runs of positions cost fewer instructions and segment look-ups, which is what counts while the launch is a chain of
// latencies: up to a million rows, at all levels, and near the root, where a thread's eight bins and its neighbours' share cache
// lines. With more rows and nodes the launch is bound by the lines it asks for, and a wave that takes 64 positions side by
// side asks for those that lie close together. Runs against positions apart, us for 1, 4, 8, 32, 128 and 512 nodes:
//   400,000 x 60          4.8 : 7.7   4.8 : 6.5   5.5 : 6.9   6.2 : 7.7   7.0 : 8.8   8.7 : 9.9
//   1,000,000 x 50        5.4 : 8.9   5.6 : 7.6   6.8 : 7.5   8.9 : 9.2   9.8 : 11.2  12.2 : 14.3
//   1,400,000 x 60        6.2 : 9.1   6.0 : 7.7   7.9 : 8.0  10.6 : 9.7  12.1 : 12.4  17.8 : 19.3
//   2,000,000 x 100       7.8 : 10.4  6.8 : 8.3   8.8 : 8.6  13.6 : 11.4 16.2 : 15.7
//   4,000,000 x 100      11.6 : 13.4 10.8 : 10.9 14.3 : 11.8 23.2 : 19.0 32.4 : 30.7
//   10,000,000 x 100     22.3 : 30.6 22.2 : 28.2 31.7 : 31.1 53.6 : 48.2 87.4 : 82.8
//   100,000,000 x 4       125 : 208   159 : 222   260 : 263   570 : 478   974 : 897
// Apart at 128 nodes or more with 100,000 x 32 (columns that one L2 holds): 8.7 : 8.4, 10.2 : 9.4 at 512.
constexpr int64_t kRunsAlways = int64_t(1) << 20;
constexpr bool classify_in_runs(int n_nodes, int64_t n_rows) { return n_nodes <= 4 || n_rows <= kRunsAlways; }

// Leaf of every row that is still in a node after the last level: the node itself if it
// did not split, else the child the row falls into.
template <typename T, typename BinT>
__global__ void __launch_bounds__(kThreads)
  final_leaf_kernel(const int32_t* __restrict__ rows, int64_t n, const int32_t* __restrict__ seg,
                    const int32_t* __restrict__ block_seg, int n_parents, int level_first, const T* X, int F,
                    const BinT* bins_t, int64_t bins_stride, const int32_t* feature, const double* split,
                    const int32_t* split_bin, int32_t* row_leaf)
{
  __shared__ int s_seg[kSegLds];
  const int64_t base    = blockIdx.x * static_cast<int64_t>(kPartBlock);
  const SlabSegments ss = load_slab_segments(seg, n_parents, block_seg, blockIdx.x, base, n, s_seg);
#pragma unroll
  for (int u = 0; u < kPartItems; u++) {
    const int64_t i = base + u * kThreads + threadIdx.x;
    if (i >= n) continue;
    const int j = segment_of(ss, s_seg, seg, static_cast<int>(i));
    if (j < 0) continue;  // retired earlier: recorded when it retired
    int node      = level_first + j;
    const int row = rows[i];
    const int ft  = feature[node];
    if (ft != -1) {
      bool left;
      if (bins_t != nullptr)
        left = static_cast<int>(bins_t[ft * bins_stride + row]) <= split_bin[node];
      else
        left = static_cast<double>(X[static_cast<int64_t>(row) * F + ft]) <= split[node];
      node = left ? left_child(node) : right_child(node);
    }
    row_leaf[row] = node;
  }
}

// The same result, written window by window of the row space. The rows of a node ascend
// along its segment (the partition is stable and starts from the identity), so the rows of
// one window [w * kLeafWindow, (w + 1) * kLeafWindow) form one contiguous run in every
// segment. A workgroup that takes all those runs writes a contiguous piece of row_leaf
// whole, where the order of the segments scatters four bytes into a different cache line per row.
constexpr int kLeafWindow   = 8192;     // rows per workgroup
constexpr int kLeafThreads  = 1024;
constexpr int kLeafParents  = 4096;     // segments a workgroup can index in its LDS
constexpr int64_t kLeafBoundsEntries = int64_t(1) << 20;

// bounds[j * (n_windows + 1) + w] = first index of segment j whose row is >= w * kLeafWindow
__global__ void __launch_bounds__(kThreads)
  leaf_window_bounds_kernel(const int32_t* __restrict__ rows, const int32_t* seg, int n_parents, int n_windows,
                            int32_t* bounds)
{
  const int64_t t = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  if (t >= static_cast<int64_t>(n_parents) * (n_windows + 1)) return;
  const int j = static_cast<int>(t / (n_windows + 1));
  const int w = static_cast<int>(t - static_cast<int64_t>(j) * (n_windows + 1));
  int lo = seg[j], hi = seg[j + 1];
  if (w == n_windows) {
    lo = hi;
  } else if (w > 0) {
    const int64_t first = static_cast<int64_t>(w) * kLeafWindow;
    while (lo < hi) {
      const int mid = lo + ((hi - lo) >> 1);
      if (rows[mid] < first)
        lo = mid + 1;
      else
        hi = mid;
    }
  }
  bounds[t] = lo;
}

template <typename BinT>
__global__ void __launch_bounds__(kLeafThreads)
  final_leaf_window_kernel(const int32_t* __restrict__ rows, const int32_t* bounds, int n_parents, int n_windows,
                           int level_first, const BinT* bins_t, int64_t bins_stride, const int32_t* feature,
                           const int32_t* split_bin, int32_t* row_leaf)
{
  __shared__ int s_lo[kLeafParents];
  __shared__ int s_pre[kLeafParents + 1];  // exclusive prefix of the run lengths
  __shared__ int s_wave[kLeafThreads / 64];
  const int w = blockIdx.x;
  // run of every segment in this window, four segments per thread
  constexpr int kPer = kLeafParents / kLeafThreads;
  int len[kPer];
  int mine = 0;
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    const int j = threadIdx.x * kPer + u;
    len[u]      = 0;
    if (j < n_parents) {
      const int32_t* b = bounds + static_cast<int64_t>(j) * (n_windows + 1) + w;
      const int lo     = b[0];
      s_lo[j]          = lo;
      len[u]           = b[1] - lo;
    }
    mine += len[u];
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int incl = mine;
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(incl, off, 64);
    if (lane >= off) incl += o;
  }
  if (lane == 63) s_wave[wave] = incl;
  __syncthreads();
  if (threadIdx.x == 0) {
    int run = 0;
    for (int i = 0; i < kLeafThreads / 64; i++) {
      const int v = s_wave[i];
      s_wave[i]   = run;
      run += v;
    }
    s_pre[n_parents] = run;
  }
  __syncthreads();
  int run = s_wave[wave] + incl - mine;
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    const int j = threadIdx.x * kPer + u;
    if (j < n_parents) s_pre[j] = run;
    run += len[u];
  }
  __syncthreads();
  const int total = s_pre[n_parents];
  for (int t = threadIdx.x; t < total; t += kLeafThreads) {
    // last segment whose prefix is <= t (empty runs share a prefix; the last of them holds t)
    int lo = 0, hi = n_parents;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (s_pre[mid] <= t)
        lo = mid;
      else
        hi = mid;
    }
    const int row = rows[s_lo[lo] + (t - s_pre[lo])];
    int node      = level_first + lo;
    const int ft  = feature[node];
    if (ft != -1)
      node = static_cast<int>(bins_t[ft * bins_stride + row]) <= split_bin[node] ? left_child(node) : right_child(node);
    row_leaf[row] = node;
  }
}

// (retired, left) counts as one 64-bit word: sums of words are sums of both
__device__ __forceinline__ int64_t pair_word(int2 c) { return (static_cast<int64_t>(c.x) << 32) + c.y; }
__device__ __forceinline__ int2 word_pair(int64_t v) { return make_int2(static_cast<int>(v >> 32), static_cast<int>(v)); }

// pass 2: the counts become prefix counts, and with them one wave per parent j finds the prefix counts at its
// segment's start, the segment starts of its two children in the next level, and for every slab of the next level's
// order that begins inside one of these children the child's number (what load_slab_segments starts from). The wave
// of parent 0 also marks the slabs that begin among the retired rows.
// Every workgroup scans all slabs' counts for itself: that is read-only work which it would otherwise wait for, a
// launch of one workgroup in front of this one. Its threads take `per` slabs each; what lies between a thread's first
// slab and a segment's start is added by the wave, the slabs' counts and then the rows' codes, 32 a lane in two loads.
// Bound by latency (a launch, the counts, the segment's start, the codes): with a kernel of its own for the scan and
// codes read one byte a lane, 1,000,000 rows took 4.6 + 13 us from 16 parents on, now 6 (10,000,000 rows: 6 + 12, now 8).
constexpr int kScanThreads = 1024;

struct SlabPrefix {
  const int64_t* s_before;  // [kScanThreads] counts of the slabs before a thread's first one
  const int2* counts;
  const uint8_t* code;
  int per;
  int64_t n, total;
};

// what the wave's lanes have to add up for the prefix counts at index s
__device__ __forceinline__ int64_t prefix_share(const SlabPrefix& p, int s, int lane)
{
  if (s >= p.n) return 0;
  const int b    = s / kPartBlock;
  const int rest = s - b * kPartBlock;
  int64_t share  = 0;
  for (int i = b / p.per * p.per + lane; i < b; i += 64) share += pair_word(p.counts[i]);
  constexpr int kBytes = kPartBlock / 64;
  static_assert(kBytes % 16 == 0, "a lane's codes are whole 16-byte pieces");
  int zeros = 0, ones = 0;
#pragma unroll
  for (int piece = 0; piece < kBytes; piece += 16) {
    const int first = lane * kBytes + piece;
    if (first < rest) {
      const uint4 v = *reinterpret_cast<const uint4*>(p.code + static_cast<int64_t>(b) * kPartBlock + first);
      const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int left      = rest - first - 4 * i;  // codes of this word in front of s; a code is 0, 1 or 2
        const unsigned mask = left >= 4 ? 0x01010101u : left <= 0 ? 0u : 0x01010101u & ((1u << (8 * left)) - 1);
        ones  += __popc(w[i] & mask);
        zeros += __popc(~(w[i] | w[i] >> 1) & mask);
      }
    }
  }
  return share + pair_word(make_int2(zeros, ones));
}
__device__ __forceinline__ int2 prefix_at(const SlabPrefix& p, int s, int64_t share)
{
  if (s >= p.n) return word_pair(p.total);
  return word_pair(p.s_before[s / kPartBlock / p.per] + wave_read_lane(wave_inclusive_sum(share), 63));
}

__global__ void __launch_bounds__(kScanThreads)
  child_segments_kernel(const int32_t* __restrict__ seg, int n_parents, int64_t n, const uint8_t* __restrict__ code,
                        const int2* __restrict__ block_counts, int n_slabs, int2* block_offsets, int2* seg_prefix,
                        int32_t* seg_next, int32_t* block_seg_next)
{
  __shared__ int64_t s_before[kScanThreads];
  __shared__ int64_t s_wave[kScanThreads / 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int j    = blockIdx.x * (kScanThreads / 64) + wave;
  const int per  = (n_slabs + kScanThreads - 1) / kScanThreads;
  const int s0   = j < n_parents ? seg[j] : 0, s1 = j < n_parents ? seg[j + 1] : 0;
  const int begin = min(n_slabs, static_cast<int>(threadIdx.x) * per), end = min(n_slabs, begin + per);
  // eight slabs at a time, so that their loads are in flight together
  constexpr int kAtOnce = 8;
  int64_t slab[kAtOnce];
  auto load_slabs = [&](int first) {
#pragma unroll
    for (int u = 0; u < kAtOnce; u++) slab[u] = first + u < end ? pair_word(block_counts[first + u]) : 0;
  };
  int64_t mine = 0;
  for (int b = begin; b < end; b += kAtOnce) {
    load_slabs(b);
#pragma unroll
    for (int u = 0; u < kAtOnce; u++) mine += slab[u];
  }
  SlabPrefix p{s_before, block_counts, code, per, n, 0};
  const int64_t share0 = prefix_share(p, s0, lane), share1 = prefix_share(p, s1, lane);
  const int64_t incl = wave_inclusive_sum(mine);
  if (lane == 63) s_wave[wave] = incl;
  __syncthreads();
  int64_t before = incl - mine;
  for (int w = 0; w < kScanThreads / 64; w++) {
    before += w < wave ? s_wave[w] : 0;
    p.total += s_wave[w];
  }
  s_before[threadIdx.x] = before;
  if (blockIdx.x == 0)
    for (int b = begin; b < end; b += kAtOnce) {
      if (per > kAtOnce) load_slabs(b);
#pragma unroll
      for (int u = 0; u < kAtOnce; u++) {
        if (b + u < end) block_offsets[b + u] = word_pair(before);
        before += slab[u];
      }
    }
  __syncthreads();
  if (j >= n_parents) return;
  const int2 p0 = prefix_at(p, s0, share0), p1 = prefix_at(p, s1, share1);
  const int total_dead = word_pair(p.total).x;
  const int left  = total_dead + (s0 - p0.x);          // start of the left child's run
  const int right = left + (p1.y - p0.y);              // start of the right child's run
  const int stop  = left + (s1 - s0) - (p1.x - p0.x);  // end of the right child's run
  if (lane == 0) {
    seg_prefix[j]       = p0;
    seg_next[2 * j]     = left;
    seg_next[2 * j + 1] = right;
    if (j == n_parents - 1) seg_next[2 * n_parents] = static_cast<int32_t>(n);
  }
  auto mark = [&](int from, int to, int value) {
    for (int64_t b = (static_cast<int64_t>(from) + kPartBlock - 1) / kPartBlock + lane; b * kPartBlock < to; b += 64)
      block_seg_next[b] = value;
  };
  if (j == 0) mark(0, total_dead, -1);
  mark(left, right, 2 * j);
  mark(right, stop, 2 * j + 1);
}

// number of set bits of a 64-bit wave mask below the calling lane
__device__ inline int prefix_popc(unsigned long long mask)
{
  return __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), 0));
}

// pass 3: scatter every row to its place in the next level's order. Rows are
// taken in slabs of one workgroup width (coalesced); inside a slab the ranks
// come from wave ballots, across waves and slabs from a 32-entry scan.
struct ScatterArgs {
  const int32_t* rows;
  int64_t n;
  const uint8_t* code;
  const int2* block_offsets;
  const int32_t* seg;
  const int32_t* block_seg;
  const int2* seg_prefix;
  const int32_t* seg_next;
  int level_first, n_parents;
  int32_t* rows_out;
  int32_t* row_leaf;
};
__device__ __forceinline__ void scatter_slab(const ScatterArgs& a, int slab)
{
  const int32_t* __restrict__ const rows      = a.rows;
  const int32_t* __restrict__ const seg       = a.seg;
  const int32_t* __restrict__ const block_seg = a.block_seg;
  const int2* const block_offsets             = a.block_offsets;
  const int2* const seg_prefix                = a.seg_prefix;
  const int32_t* const seg_next               = a.seg_next;
  const uint8_t* const code                   = a.code;
  int32_t* const rows_out                     = a.rows_out;
  int32_t* const row_leaf                     = a.row_leaf;
  const int64_t n                             = a.n;
  const int level_first = a.level_first, n_parents = a.n_parents;
  constexpr int kWaves = kThreads / 64;
  __shared__ int s_seg[kSegLds];
  __shared__ int s_cnt[kPartItems * kWaves];  // retired << 16 | left, in row order
  const int64_t base = slab * static_cast<int64_t>(kPartBlock);
  const int wave     = threadIdx.x >> 6;
  int row[kPartItems];
  int c[kPartItems];
  int below_d[kPartItems], below_l[kPartItems];
  // rows and codes are requested before the slab's segments, which they do not depend on
#pragma unroll
  for (int u = 0; u < kPartItems; u++) {
    int64_t i = base + u * kThreads + threadIdx.x;
    c[u]      = 3;
    row[u]    = 0;
    if (i < n) {
      row[u] = rows[i];
      c[u]   = code[i];
    }
  }
  const SlabSegments ss = load_slab_segments(seg, n_parents, block_seg, slab, base, n, s_seg);
  const int2 boff       = block_offsets[slab];
  // Per row: its segment and what its destination is counted from. A left row goes to
  // seg_next[2j] + (left rows of the segment before it), a right row to seg_next[2j+1] + (right
  // rows of the segment before it); both counts are differences of prefix counts, whose
  // segment-start part is known here already.
  int seg_j[kPartItems], dbase[kPartItems];
#pragma unroll
  for (int u = 0; u < kPartItems; u++) {
    const int64_t i = base + u * kThreads + threadIdx.x;
    seg_j[u]        = i < n ? segment_of(ss, s_seg, seg, static_cast<int>(i)) : -1;
    dbase[u]        = 0;
    if (c[u] == 1 || c[u] == 2) {
      const int j   = seg_j[u];
      const int2 sp = seg_prefix[j];
      dbase[u]      = c[u] == 1 ? seg_next[2 * j] - sp.y : seg_next[2 * j + 1] - (seg[j] - sp.x - sp.y);
    }
  }
#pragma unroll
  for (int u = 0; u < kPartItems; u++) {
    unsigned long long md = __ballot(c[u] == 0);
    unsigned long long ml = __ballot(c[u] == 1);
    below_d[u]            = prefix_popc(md);
    below_l[u]            = prefix_popc(ml);
    if ((threadIdx.x & 63) == 0) s_cnt[u * kWaves + wave] = (__popcll(md) << 16) | __popcll(ml);
  }
  __syncthreads();
  // exclusive scan of the kPartItems * kWaves = 32 counts by one wave
  static_assert(kPartItems * kWaves <= 64, "one wave scans the slab's counts");
  if (wave == 0) {
    const int lane = threadIdx.x;
    const int v    = lane < kPartItems * kWaves ? s_cnt[lane] : 0;
    int incl       = v;
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(incl, off, 64);
      if (lane >= off) incl += o;
    }
    if (lane < kPartItems * kWaves) s_cnt[lane] = incl - v;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPartItems; u++) {
    int64_t i = base + u * kThreads + threadIdx.x;
    if (i < n) {
      const int excl = s_cnt[u * kWaves + wave];
      const int D    = boff.x + (excl >> 16) + below_d[u];
      const int L    = boff.y + (excl & 0xffff) + below_l[u];
      int dest;
      if (c[u] == 0) {
        dest = D;
        // a row that retires now sits in a leaf: remember which
        if (row_leaf != nullptr && seg_j[u] >= 0) row_leaf[row[u]] = level_first + seg_j[u];
      } else if (c[u] == 1) {
        dest = dbase[u] + L;
      } else {
        dest = dbase[u] + (static_cast<int>(i) - D - L);
      }
      rows_out[dest] = row[u];
    }
  }
}

__global__ void __launch_bounds__(kThreads) scatter_kernel(ScatterArgs a) { scatter_slab(a, blockIdx.x); }

// What a level begins with, in one launch: its rows in their places, the tiles of its built nodes, and their histograms cleared. None of the
// three waits for another; as launches of their own the tiles were 5 us and a gap behind every scatter, the clearing 6 to 65. With that and the
// splits applied where rows are classified, kernels of a tree and their gaps, us: 1,000,000 x 50 depth 12 with 512 samples 1582 -> 1498, 1,000,000 x 60
// with 3 outputs depth 10 1708 -> 1598, 2,000,000 x 120 depth 8 1696 -> 1617; 10,000,000 x 100, whose scatter is bound by memory, as before.
__global__ void __launch_bounds__(kThreads) level_start_kernel(PlanArgs plan, ScatterArgs scatter, int n_slabs, int clear_from, int clear_parts)
{
  static_assert(kThreads == kPlanThreads, "one size of workgroup");
  int block = blockIdx.x;
  const int plan_blocks = (plan.blocks + 7) / 8 * 8;  // a slab stays with the XCD whose L2 has its rows and codes
  if (block < plan_blocks) {
    if (block < plan.blocks) plan_tiles_block(plan, block);
    return;
  }
  block -= plan_blocks;
  if (block < n_slabs) return scatter_slab(scatter, block);
  block -= n_slabs;
  clear_built(plan.hist, plan.node_sums, clear_from + block / clear_parts, block % clear_parts, clear_parts);
}

// The reference's (node, row) pairs, for the observation points: node of the level that the
// order belongs to, -1 for retired rows.
__global__ void __launch_bounds__(kThreads)
  expand_positions_kernel(const int32_t* __restrict__ rows, int64_t n, const int32_t* __restrict__ seg,
                          const int32_t* __restrict__ block_seg, int n_parents, int level_first, int2* out)
{
  __shared__ int s_seg[kSegLds];
  const int64_t base    = blockIdx.x * static_cast<int64_t>(kPartBlock);
  const SlabSegments ss = load_slab_segments(seg, n_parents, block_seg, blockIdx.x, base, n, s_seg);
#pragma unroll
  for (int u = 0; u < kPartItems; u++) {
    const int64_t i = base + u * kThreads + threadIdx.x;
    if (i >= n) continue;
    const int j = segment_of(ss, s_seg, seg, static_cast<int>(i));
    out[i]      = make_int2(j >= 0 ? level_first + j : -1, rows[i]);
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

struct Layout {
  // tree state
  I64Pair* node_sums;
  uint8_t* tainted;
  double* scales;
  unsigned long long* qstats;
  // proposals
  void* uniq;
  int32_t* counts;
  void* proposals;
  double* proposals_d;
  int32_t* row_pointers;
  int32_t* bin_feature;
  void* upload_block;
  size_t upload_bytes;
  int32_t* groups;
  int32_t* sgroups;
  int2* bin_lanes;
  RecInfo* rec;
  void* binned;
  size_t binned_bytes;
  uint2* tables;
  void* map_x;
  float* map_t;
  int32_t* straight;
  // quantiser
  double* part_a[2];
  double* part_b[2];
  int2* qgh;
  // positions: row numbers in node order, segment starts, first segment of every slab
  int32_t* rows[2];
  int32_t* seg[2];
  int32_t* block_seg[2];
  uint8_t* code;
  int32_t* split_bin;
  void* bins_t;
  int64_t bins_t_stride;
  int2* block_counts;
  int2* block_offsets;
  int2* seg_prefix;
  int32_t* leaf_bounds;
  // histogram
  int32_t* tile_start;
  int4* tiles;
  LevelMeta* meta;
  int32_t* pair_sync;
  unsigned long long* partials;
  int32_t* partial_lists;
  int32_t* partial_list_count;
  int32_t* partial_count;
  LevelMeta* level_totals;
  Cand* partial;
  I64Pair* hist;
  size_t hist_bytes;
  I64Pair* left;  // left sums of the candidates of a level without histograms in memory; null: no such levels
  // null pointers when the shape is not one for these builders
  SmallTreeState small;
  MidTreeState mid;
};

// Room for the histograms of all levels, where the caller leaves the budget to the library: a 64th of the memory.
constexpr double kWholeTreeBytes = 4.5e9;

// The bytes of histograms a build may keep (where one node needs more: that node's). roomy: see build_tree_impl,
// where a level that outgrows the reference's budget keeps its parents
double hist_budget(int64_t cache_bytes, bool roomy)
{
  return cache_bytes > 0 ? static_cast<double>(cache_bytes) : (roomy ? kWholeTreeBytes : 1e9);
}
size_t hist_bytes_bound(int F, int K, int S, int max_depth, int64_t cache_bytes, bool roomy)
{
  if (max_depth < 1) return 0;
  const double bpn = static_cast<double>(K) * F * S * 16.0;  // bytes per node with every bin distinct
  double a = std::max(hist_budget(cache_bytes, roomy), bpn);
  double b = static_cast<double>(level_end(max_depth - 1)) * bpn;
  return static_cast<size_t>(std::min(a, b)) + 256;
}

void make_layout(Arena& ar, Layout& L, int64_t N, int F, int K, int max_depth, int S,
                 size_t elem, int64_t cache_bytes, bool roomy)
{
  const int64_t max_nodes   = level_end(max_depth);
  const int64_t level_nodes = int64_t(1) << (max_depth > 0 ? max_depth - 1 : 0);
  L.node_sums    = ar.take<I64Pair>(max_nodes * K);
  L.tainted      = ar.take<uint8_t>(max_nodes);
  L.scales       = ar.take<double>(4);
  L.qstats       = ar.take<unsigned long long>(2);
  L.uniq         = ar.take<char>(static_cast<size_t>(F) * S * elem);
  L.counts       = ar.take<int32_t>(F);
  L.proposals    = ar.take<char>(static_cast<size_t>(F) * S * elem);
  L.proposals_d  = ar.take<double>(static_cast<size_t>(F) * S);
  L.row_pointers = ar.take<int32_t>(F + 1);
  L.bin_feature  = ar.take<int32_t>(static_cast<size_t>(F) * S);
  // the tables hist_prepare sends from the host: one block, filled by one copy
  const size_t upload_at = ar.used;
  L.groups       = ar.take<int32_t>(F + 1);
  L.sgroups      = ar.take<int32_t>(F + 1);
  L.bin_lanes    = ar.take<int2>(bin_lanes_max(F));
  L.rec          = ar.take<RecInfo>(F);
  L.upload_block = L.groups;
  L.upload_bytes = ar.used - upload_at;
  // bin cache: one or two bytes per (row, feature); used when the tree has at least two levels
  L.binned_bytes = max_depth >= 2 ? bin_cache_bytes(N, F, S) : 0;
  L.binned       = max_depth >= 2 ? static_cast<void*>(ar.take<char>(L.binned_bytes + 16)) : nullptr;
  L.tables       = ar.take<uint2>(2 * static_cast<size_t>(F) * kMaxCells / 32);
  L.map_x        = ar.take<double>(4 * static_cast<size_t>(F));
  L.map_t        = ar.take<float>(2 * static_cast<size_t>(F));
  L.straight     = ar.take<int32_t>(F);
  int64_t n_chunks = (N * K + 4095) / 4096;
  for (int i = 0; i < 2; i++) {
    L.part_a[i] = ar.take<double>(n_chunks);
    L.part_b[i] = ar.take<double>(n_chunks);
    n_chunks    = (n_chunks + 4095) / 4096;
  }
  L.qgh    = ar.take<int2>(N * K);
  L.rows[0] = ar.take<int32_t>(N);
  L.rows[1] = ar.take<int32_t>(N);
  L.seg[0]  = ar.take<int32_t>(level_nodes + 1);
  L.seg[1]  = ar.take<int32_t>(level_nodes + 1);
  L.block_seg[0] = ar.take<int32_t>((N + kPartBlock - 1) / kPartBlock);
  L.block_seg[1] = ar.take<int32_t>((N + kPartBlock - 1) / kPartBlock);
  L.code   = ar.take<uint8_t>(N);
  L.split_bin = ar.take<int32_t>(max_nodes);
  // feature-major bins for the position update (needs the bin cache)
  L.bins_t_stride = (N + kTransRows - 1) / kTransRows * kTransRows;
  L.bins_t = max_depth >= 2 ? static_cast<void*>(ar.take<char>(static_cast<size_t>(F) * L.bins_t_stride * (S <= 256 ? 1 : 2)))
                            : nullptr;
  const int64_t n_pblocks = (N + kPartBlock - 1) / kPartBlock;
  L.block_counts  = ar.take<int2>(n_pblocks);
  L.block_offsets = ar.take<int2>(n_pblocks);
  L.seg_prefix    = ar.take<int2>(level_nodes);
  L.leaf_bounds   = max_depth >= 2 ? ar.take<int32_t>(kLeafBoundsEntries) : nullptr;
  L.tile_start    = ar.take<int32_t>(level_nodes + 1);
  // a tile holds at least 8 rows (two rows per pass, four passes); every node adds at most one partial tile
  L.tiles         = ar.take<int4>(N / 8 + level_nodes + 1);
  L.meta          = ar.take<LevelMeta>(1);
  L.pair_sync     = ar.take<int32_t>(kPairSyncSlots);
  // parked sub-histograms of a launch on cached bins (kPartialSlots of the widest group the LDS can hold)
  L.partials      = max_depth >= 2 ? ar.take<unsigned long long>(static_cast<size_t>(kPartialSlots) * kPartialStrideMax)
                                   : nullptr;
  L.partial_lists = ar.take<int32_t>(static_cast<size_t>(kPartialMaxLists) * kPartialListCap);
  L.partial_list_count = ar.take<int32_t>(kPartialMaxLists);
  L.partial_count = ar.take<int32_t>(1);
  L.level_totals  = ar.take<LevelMeta>(max_depth > 0 ? max_depth : 1);
  // candidates per node: one per chunk of bins (split_eval_kernel) or one per feature (scan_split_kernel)
  const int64_t max_chunks = std::max<int64_t>((static_cast<int64_t>(F) * S + kSplitChunk - 1) / kSplitChunk, F);
  L.partial       = ar.take<Cand>(level_nodes * max_chunks);
  L.left          = K == 1 && max_depth >= 2 && S <= kDirectMaxBins ? ar.take<I64Pair>(level_nodes * F) : nullptr;
  // one of the builders at a time uses the room for histograms
  const size_t mid_bytes = mid_tree_fits(N, F, K, max_depth, S) ? mid_hist_bytes(N, F, K, max_depth, S) : 0;
  // (counted with 16 bytes a bin: with a budget between that and the 8 it takes, its other arrays would need more than a tree one level
  // deeper, which is not its size, does in all)
  const double mid_counted = static_cast<double>(mid_bytes) + 2.0 * level_nodes * K * F * S * 8;
  bool mid = mid_bytes > 0 && mid_counted <= hist_budget(cache_bytes, roomy);
  const bool small       = small_tree_fits(N, F, K, max_depth, S) && !(mid && mid_beats_small(N, F, K, max_depth, S));
  mid                    = mid && !small;
  L.hist_bytes        = hist_bytes_bound(F, K, S, max_depth, cache_bytes, roomy);
  char* const hist    = ar.take<char>(std::max(L.hist_bytes, mid ? mid_bytes : 0));
  L.hist              = reinterpret_cast<I64Pair*>(hist);
  L.small = SmallTreeState{};
  if (small) {
    SmallTreeState& st    = L.small;
    st.pitch              = (N + 7) / 8 * 8;
    const size_t per_row  = static_cast<size_t>(F) * st.pitch;
    st.order[0]    = ar.take<uint32_t>(per_row);
    st.order[1]    = ar.take<uint32_t>(per_row);
    st.bins        = ar.take<uint16_t>(per_row);
    st.proposals   = ar.take<double>(static_cast<size_t>(F) * S);
    st.counts      = ar.take<int32_t>(F);
    st.rp          = ar.take<int32_t>(F);
    for (auto& nodes : st.node_of_pos) nodes = ar.take<uint16_t>(st.pitch);
    st.code        = ar.take<uint8_t>(st.pitch);
    st.seg         = ar.take<int2>(max_nodes);
    st.live        = ar.take<int32_t>(max_depth + 1);
    st.base        = ar.take<I64Pair>(max_nodes * K);
    st.node_sums   = L.node_sums;
    st.qgh         = L.qgh;
    st.scales      = L.scales;
    const bool decides = K == 1 && F <= kSmallDecideFeatures;
    st.cand[0]     = ar.take<SmallCand>(level_nodes * F);
    st.cand[1]     = decides ? ar.take<SmallCand>(level_nodes * F) : st.cand[0];
    if (small_tree_levels_fit(N, F, K, max_depth)) {
      st.sync  = ar.take<uint32_t>(kSmallDecideFeatures);
      st.found = ar.take<unsigned long long>(3 * (2 * level_nodes - 1) * F);
    }
    for (auto& left : st.left) left = decides ? ar.take<I64Pair>(level_nodes * F) : nullptr;
  }
  L.mid = MidTreeState{};
  if (mid) {
    MidTreeState& st   = L.mid;
    st.pitch           = (N + 255) / 256 * 256;
    st.bin_bytes       = S <= 256 ? 1 : 2;
    const size_t fs    = static_cast<size_t>(F) * S;
    const size_t level_hist = static_cast<size_t>(level_nodes) * K * fs;
    st.bins       = ar.take<char>(static_cast<size_t>(F) * st.pitch * st.bin_bytes);
    st.props      = ar.take<char>(fs * elem);
    st.proposals  = ar.take<double>(fs);
    st.cells      = 128;  // eight cells per proposal
    while (st.cells < 8 * S && st.cells < kMaxCells) st.cells *= 2;
    st.tables     = ar.take<uint2>(static_cast<size_t>(F) * st.cells / 32);
    st.map_x      = ar.take<char>(2 * static_cast<size_t>(F) * elem);
    st.map_t      = ar.take<float>(2 * static_cast<size_t>(F));
    st.counts     = ar.take<int32_t>(F);
    st.rp         = ar.take<int32_t>(F + 1);
    st.chunk_sums = ar.take<double>(2 * ((N * K + 4095) / 4096));
    st.q          = ar.take<int2>(static_cast<size_t>(K) * st.pitch);
    for (auto& nodes : st.row_node) nodes = ar.take<uint16_t>(st.pitch);
    st.q_stats    = ar.take<unsigned long long>(4);
    if (hist != nullptr) {
      st.hist[0]  = reinterpret_cast<uint2*>(L.hist);
      st.hist[1]  = st.hist[0] + level_hist;
      st.images   = reinterpret_cast<unsigned long long*>(st.hist[0] + 2 * level_hist);
    }
    st.node_sums  = L.node_sums;
    st.scales     = L.scales;
    st.cand       = ar.take<SmallCand>(level_nodes * F);
    st.left       = ar.take<uint2>(level_nodes * F);
    st.splits     = ar.take<int2>(level_nodes);
    st.live       = ar.take<int32_t>(max_depth + 1);
  }
}

int validate(int64_t N, int F, int K, const lbt_build_params* p, int x_dtype)
{
  LBT_REQUIRE(p != nullptr, "params is null");
  LBT_REQUIRE(p->struct_bytes == static_cast<int32_t>(sizeof(lbt_build_params)),
              "lbt_build_params.struct_bytes is %d, this library's struct has %d bytes: set it to "
              "sizeof(lbt_build_params) of the lbtree.h the library was built with, in a zero-initialised struct",
              p->struct_bytes, static_cast<int>(sizeof(lbt_build_params)));
  LBT_REQUIRE(x_dtype == LBT_F32 || x_dtype == LBT_F64, "unsupported X dtype %d", x_dtype);
  LBT_REQUIRE(N >= 1 && N < 2147483647LL, "n_rows %lld out of range", static_cast<long long>(N));
  LBT_REQUIRE(F >= 1 && K >= 1, "n_features and n_outputs must be positive");
  LBT_REQUIRE(K <= 65535, "n_outputs above 65535 is not supported");
  LBT_REQUIRE(p->max_depth >= 0 && p->max_depth <= 24, "max_depth %d out of range [0,24]", p->max_depth);
  LBT_REQUIRE(static_cast<int64_t>(p->max_nodes) == level_end(p->max_depth),
              "max_nodes must be 2^(max_depth+1)-1");
  LBT_REQUIRE(p->split_samples >= 1 && p->split_samples <= LBT_MAX_SPLIT_SAMPLES,
              "split_samples must be in [1, %d]", LBT_MAX_SPLIT_SAMPLES);
  LBT_REQUIRE(p->dataset_rows >= 1, "dataset_rows must be positive");
  LBT_REQUIRE(p->hist_cache_bytes >= 0, "hist_cache_bytes must not be negative");
  return LBT_OK;
}


// What the host reads back in the middle of a call (bin counts per feature, the quantiser's
// overflow flag): pinned memory and two events per host thread, so that each value is waited
// for by itself and not together with everything else that is queued on the stream.
int host_mirror(int F, ThreadResources** out)
{
  ThreadResources* here = nullptr;
  LBT_TRY(thread_resources_here(&here));
  ThreadResources& hm = *here;
  if (hm.counts_here == nullptr) LBT_HIP(hipEventCreateWithFlags(&hm.counts_here, hipEventDisableTiming));
  if (hm.stats_here == nullptr) LBT_HIP(hipEventCreateWithFlags(&hm.stats_here, hipEventDisableTiming));
  // an earlier call of this thread that did not wait (or failed half-way) may still own the buffer
  LBT_HIP(hipEventSynchronize(hm.counts_here));
  LBT_HIP(hipEventSynchronize(hm.stats_here));
  const size_t need = static_cast<size_t>(F) + 1;
  if (hm.mirror_capacity < need) {
    if (hm.mirror != nullptr) LBT_HIP(hipHostFree(hm.mirror));
    hm.mirror          = nullptr;
    hm.mirror_capacity = 0;
    LBT_HIP(hipHostMalloc(reinterpret_cast<void**>(&hm.mirror), sizeof(int32_t) * (4 + need), hipHostMallocDefault));
    hm.mirror_capacity = need;
  }
  *out = &hm;
  return LBT_OK;
}

// SelectSplitSamples (build_tree.cu:867-964) and what the quantiser rounds with (build_tree.cu:51-140): the two absolute sums in a
// fixed order, the scales. Without samples (F = 0) or without sums (sums.scales null) only the other one. first_level: the chunk
// sums of |g| and |h| if the caller has them already ([2][chunks], see lbt_weighted_gradient_sums), else null.
// part_a/part_b: two levels of partial sums.
template <typename T>
int start_tree(hipStream_t stream, SampleArgs<T> samples, const InitArgs* init, const double* g, const double* h, int64_t n,
               double* const (&part_a)[2], double* const (&part_b)[2], double* scales, unsigned long long* qstats,
               const double* first_level)
{
  samples.P = 2;
  while (samples.P < samples.S) samples.P <<= 1;
  int64_t m = (n + kSumChunk - 1) / kSumChunk;
  SumArgs sums{};
  if (scales != nullptr) {
    sums = SumArgs{g, h, n, first_level != nullptr ? 0 : static_cast<int>(m), {part_a[0], part_b[0]}, {part_a[0], part_b[0]}, 0, scales, qstats};
    if (first_level != nullptr) sums.of[0] = first_level, sums.of[1] = first_level + m;
  }
  const int64_t n_init = init == nullptr ? 0 : (std::max({init->max_nodes * init->K, init->n, init->n_slabs, static_cast<int64_t>(init->n_totals16)}) + kThreads - 1) / kThreads;
  const int64_t grid   = (samples.F + 7) / 8 * 8 + sums.m + n_init;
  if (grid > 0)
    tree_start_kernel<T><<<static_cast<unsigned>(grid), kThreads, samples.F > 0 ? samples.P * sizeof(typename KeyOf<T>::type) : 0, stream>>>(
      samples, sums, init != nullptr ? *init : InitArgs{});
  int cur = 0;
  if (scales != nullptr) {
    for (; m > kSumChunk; m = (m + kSumChunk - 1) / kSumChunk) {
      sum_level_kernel<<<static_cast<unsigned>((m + kSumChunk - 1) / kSumChunk), kThreads, 0, stream>>>(sums.of[0], sums.of[1], m, part_a[cur ^ 1],
                                                                                                        part_b[cur ^ 1]);
      cur ^= 1;
      sums.of[0] = part_a[cur];
      sums.of[1] = part_b[cur];
    }
    sums.n_of = static_cast<int>(m);
  }
  const int run    = std::max(0, samples.F - 1) / kPlaceGroups + 1;  // features of a workgroup
  const int placed = samples.F > 0 ? (samples.F - 1) / run + 1 : 0;
  tree_scales_kernel<T><<<static_cast<unsigned>(placed + (scales != nullptr ? 1 : 0)), kThreads, 0, stream>>>(samples, run, sums);
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

// GradientQuantiser and reduce_base_sums (build_tree.cu:112-129, :168-204): one rounding per (row, output), and the sums of the
// rounded pairs added to root_sums[k] (which the caller has cleared).
int round_gradients(hipStream_t stream, const double* g, const double* h, int64_t N, int K, int64_t row_offset, int32_t seed,
                    const double* scales, unsigned long long* qstats, int2* qgh, I64Pair* root_sums)
{
  auto blocks = [](int64_t n, int t) { return static_cast<unsigned>((n + t - 1) / t); };
  if (K > 1 && K <= kQuantiseFlatMaxK) {
    const unsigned gx = std::max<unsigned>(std::min<unsigned>(blocks(N * K, kQuantiseThreads), kQuantiseGroups), blocks(K, kQuantiseThreads));
    quantise_flat_kernel<<<gx, kQuantiseThreads, 2 * K * sizeof(unsigned long long), stream>>>(
      g, h, N, K, row_offset, static_cast<int64_t>(seed), scales, qgh, root_sums, qstats);
  } else {
    dim3 grid(std::min<unsigned>(blocks(N, kQuantiseThreads), kQuantiseGroups), K);
    quantise_kernel<<<grid, kQuantiseThreads, 0, stream>>>(g, h, N, K, row_offset, static_cast<int64_t>(seed), scales, qgh,
                                                   root_sums, qstats);
  }
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

// Both for the stages that want nothing else.
int run_quantiser(hipStream_t stream, const double* g, const double* h, int64_t N, int K, int64_t row_offset,
                  int32_t seed, double* const (&part_a)[2], double* const (&part_b)[2], double* scales,
                  unsigned long long* qstats, int2* qgh, I64Pair* root_sums)
{
  LBT_TRY(start_tree<float>(stream, SampleArgs<float>{}, nullptr, g, h, N * K, part_a, part_b, scales, qstats, nullptr));
  return round_gradients(stream, g, h, N, K, row_offset, seed, scales, qstats, qgh, root_sums);
}
template <typename T>
int run_split_samples(hipStream_t stream, const SampleArgs<T>& samples)
{
  double* const none[2] = {nullptr, nullptr};
  return start_tree<T>(stream, samples, nullptr, nullptr, nullptr, 0, none, none, nullptr, nullptr, nullptr);
}

// Hands the level counts of a build to the profiler: copied to the host in stream order.
int profile_levels(hipStream_t stream, const LevelMeta* totals, int max_depth, double per_row, double per_node,
                   double root_extra)
{
  static_assert(sizeof(LevelMeta) == sizeof(LevelCounts), "the host mirror of LevelMeta");
  ProfLevels* const levels = profiler().begin_levels(std::min(max_depth, 64), per_row, per_node, root_extra);
  if (levels == nullptr) return LBT_OK;
  LBT_HIP(hipMemcpyAsync(levels->host, totals, sizeof(LevelMeta) * levels->levels, hipMemcpyDeviceToHost, stream));
  LBT_HIP(hipEventRecord(levels->arrived, stream));
  return LBT_OK;
}

// The nodes whose histograms the level loop below ends up with (GetHistogram, build_tree.cu:1191-1205).
void final_histogram_range(int K, int B, const lbt_build_params& prm, int32_t* begin, int32_t* end)
{
  const uint64_t max_bytes = prm.hist_cache_bytes > 0 ? static_cast<uint64_t>(prm.hist_cache_bytes) : 1000000000ULL;
  const int64_t nodes      = static_cast<int64_t>(std::max<uint64_t>(1, max_bytes / (static_cast<uint64_t>(K) * B * 16ULL)));
  int cdepth = 0;
  while (level_end(cdepth + 1) <= nodes && cdepth <= prm.max_depth) cdepth++;
  const int64_t used_end = prm.max_depth > 0 ? level_end(prm.max_depth - 1) : 0;
  const int64_t batch    = static_cast<int64_t>(static_cast<int>(nodes));
  int64_t lo = 0, hi = level_end(cdepth);
  for (int d = 0; d < prm.max_depth; d++) {
    const int64_t in_level = int64_t(1) << d;
    for (int64_t j0 = 0; j0 < in_level; j0 += batch) {
      const int64_t b0 = level_begin(d) + j0, b1 = level_begin(d) + std::min(j0 + batch, in_level);
      if (!(b0 >= lo && b1 <= hi)) lo = b0, hi = b1;
    }
  }
  *begin = static_cast<int32_t>(lo);
  *end   = static_cast<int32_t>(std::max<int64_t>(lo, std::min<int64_t>(hi, used_end)));
}

// No observation point but the rows' leaves is asked for.
bool observes_nothing(const lbt_build_taps* t)
{
  return t == nullptr ||
         !(t->proposals || t->row_pointers || t->quantised || t->node_sums || t->positions || t->positions_per_level ||
           t->histogram || t->level_instances || t->level_built_instances || t->level_built_nodes);
}

template <typename T>
int build_tree_impl(hipStream_t stream, const T* X, int64_t row_offset, int64_t N, int F,
                    const double* g, const double* h, int K, const uint8_t* feature_set,
                    const lbt_build_params& prm, double* leaf, int32_t* feature, double* split,
                    double* gain, double* hessian, Layout& L, lbt_build_taps* taps, bool sync_at_end)
{
  const int max_depth = prm.max_depth;
  const int max_nodes = prm.max_nodes;
  const int S         = prm.split_samples;
  auto blocks = [](int64_t n, int t) { return static_cast<unsigned>((n + t - 1) / t); };

  // ---- state, split proposals, scales
  ThreadResources* hm = nullptr;
  LBT_TRY(host_mirror(F, &hm));
  int32_t* const rp_here = hm->mirror + 4;
  {
    ProfScope ps(LBT_PROF_PROPOSALS, stream);
    static_assert(sizeof(LevelMeta) == 32, "LevelMeta is cleared in 16-byte units");
    const InitArgs init{leaf, feature, split, gain, L.node_sums, max_nodes, K, L.rows[0], N, L.seg[0], L.block_seg[0], (N + kPartBlock - 1) / kPartBlock,
                        reinterpret_cast<uint4*>(L.level_totals), std::max(0, max_depth * 2), L.tainted};
    LBT_TRY(start_tree<T>(stream,
                          SampleArgs<T>{X, row_offset, N, prm.dataset_rows, F, S, 0, prm.seed, static_cast<T*>(L.uniq), L.counts, L.row_pointers,
                                        static_cast<T*>(L.proposals), L.bin_feature, L.proposals_d, F <= kMirrorFeatures ? rp_here : nullptr},
                          &init, g, h, N * K, L.part_a, L.part_b, L.scales, L.qstats, prm.abs_sum_chunks));
    if (F > kMirrorFeatures)
      LBT_HIP(hipMemcpyAsync(rp_here, L.row_pointers, sizeof(int32_t) * (F + 1), hipMemcpyDeviceToHost, stream));
    LBT_HIP(hipEventRecord(hm->counts_here, stream));
  }
  // ---- quantiser
  {
    ProfScope ps(LBT_PROF_QUANTISE, stream, static_cast<double>(N) * K * (16 + 16 + 8));
    LBT_TRY(round_gradients(stream, g, h, N, K, row_offset, prm.seed, L.scales, L.qstats, L.qgh, L.node_sums));
  }
  const unsigned long long* const h_qstats = reinterpret_cast<const unsigned long long*>(hm->mirror);
  bool stats_checked = false;
  // a gradient that does not fit 32 bits ends the call; asked once a level's work is queued,
  // when the answer has long arrived
  auto check_stats = [&]() -> int {
    if (stats_checked) return LBT_OK;
    stats_checked = true;
    LBT_HIP(hipEventSynchronize(hm->stats_here));
    if ((h_qstats[1] & kQuantTooLarge) != 0) {
      set_error("a quantised gradient or hessian reaches 2^31 and does not fit the packed 32-bit form: one entry "
                "holds the whole absolute sum and was rounded up");
      return LBT_ERR_UNSUPPORTED;
    }
    return LBT_OK;
  };

  // ---- positions and histogram cache (TreeBuilder ctor, build_tree.cu:997-1017)

  // the one host wait before the levels: the bin counts decide the feature groups. Only the
  // copy of the counts is waited for; the quantiser queued behind it keeps the GPU busy while
  // the host plans and queues the levels.
  LBT_HIP(hipEventSynchronize(hm->counts_here));
  const std::vector<int32_t> rp(rp_here, rp_here + F + 1);
  const int B = rp[F];

  HistSetup hs;
  hs.groups     = L.groups;
  hs.sgroups    = L.sgroups;
  hs.tables     = L.tables;
  hs.map_x      = L.map_x;
  hs.map_t      = L.map_t;
  hs.straight   = L.straight;
  hs.tile_start = L.tile_start;
  hs.tiles      = L.tiles;
  hs.binned     = L.binned;
  hs.binned_capacity = L.binned_bytes;
  hs.bin_lanes  = L.bin_lanes;
  hs.rec        = L.rec;
  hs.upload_block = L.upload_block;
  hs.upload_bytes = L.upload_bytes;
  // feature-major bins for the position updates of levels 0 .. max_depth-2 (and the final leaves)
  hs.bins_t        = L.binned != nullptr ? L.bins_t : nullptr;
  hs.bins_t_stride = L.bins_t_stride;
  hs.meta       = L.meta;
  hs.pair_sync  = L.pair_sync;
  hs.partials      = L.partials;
  hs.partial_lists = L.partial_lists;
  hs.partial_list_count = L.partial_list_count;
  hs.partial_count = L.partial_count;
  hs.partial_slots = kPartialSlots;
  const uint64_t max_bytes = prm.hist_cache_bytes > 0 ? static_cast<uint64_t>(prm.hist_cache_bytes) : 1000000000ULL;
  const uint64_t bytes_per_node = static_cast<uint64_t>(K) * B * 16ULL;
  uint64_t max_histogram_nodes  = std::max<uint64_t>(1, max_bytes / bytes_per_node);
  int cdepth = 0;
  while (static_cast<uint64_t>(level_end(cdepth + 1)) <= max_histogram_nodes && cdepth <= max_depth) cdepth++;
  const int64_t max_batch_size = static_cast<int64_t>(static_cast<int>(max_histogram_nodes));
  // only nodes of levels < max_depth ever get a histogram
  const int64_t used_end = max_depth > 0 ? level_end(max_depth - 1) : 0;
  HistView hv{L.hist, 0, static_cast<int>(level_end(cdepth)), K, B, nullptr};
  // histograms [node_begin, node_end): where they begin and their 16-byte units
  auto hist_range = [&](int node_begin, int node_end, uint4** begin, int64_t* n16) -> int {
    const int64_t nodes = std::max<int64_t>(std::min<int64_t>(node_end, used_end) - node_begin, 0);
    const uint64_t bytes = static_cast<uint64_t>(nodes) * bytes_per_node;
    const uint64_t skip = static_cast<uint64_t>(node_begin - hv.node_begin) * bytes_per_node;
    if (nodes > 0 && skip + bytes > L.hist_bytes) {
      set_error("histogram workspace too small (%llu > %llu)", (unsigned long long)bytes,
                (unsigned long long)L.hist_bytes);
      return LBT_ERR_WORKSPACE;
    }
    *begin = reinterpret_cast<uint4*>(reinterpret_cast<char*>(L.hist) + skip);
    *n16   = static_cast<int64_t>(bytes / 16);
    return LBT_OK;
  };
  auto zero_hist = [&](int node_begin, int node_end) -> int {
    uint4* begin = nullptr;
    int64_t n16  = 0;
    LBT_TRY(hist_range(node_begin, node_end, &begin, &n16));
    if (n16 == 0) return LBT_OK;
    ProfScope ps(LBT_PROF_OTHER, stream, 16.0 * static_cast<double>(n16));
    zero_kernel<<<static_cast<unsigned>(std::min<int64_t>((n16 + kThreads - 1) / kThreads, 65536)), kThreads, 0, stream>>>(begin, n16);
    return LBT_OK;
  };
  // Where no entry's rounded hessian is negative (known after the root's launches are queued) the children of a split have
  // a positive sum of hessians in every output, and every bin of a level is written by its scan. Two things follow for calls
  // that observe no histograms:
  //  - A level's histograms are cleared when it is reached, and only of the built siblings.
  //  - A level that outgrows the reference's 1e9 bytes does not start an empty buffer (which would make
  //    it accumulate both siblings from all rows), if the workspace has room behind its parents.
  // 2,000,000 x 200, 8 outputs, depth 8: last level 1283 -> 509 us, clearing 182 -> 90 us, the round 7.2 -> 6.4 ms.
  // Where all are positive a scanned histogram is the running sums everywhere, and any choice of built siblings gives the same
  // tree. Where some are zero (`strict`; a rare class has such) the rule on unscanned bins (build_tree.cu:645) leaves the row sum of a
  // bin in place of a running sum whose hessians are zero and whose grads are not positive. No split falls on such a bin of the node itself, nor on the
  // same bin of a descendant, where the hessians left of it are zero as well. But a sibling derived from the node differs by it from what its
  // rows add up to, and so do histograms derived from that one: the scans mark those (`tainted`). Levels in the reference's first
  // buffer are built and derived as the reference does it. A later level, which the reference adds up from all rows, derives
  // its siblings from the running sums themselves, and builds both where their parent is tainted: the same splits. Last level of three trees of
  // 2,000,000 x 200 with 8 classes, one of 0.06 %: 1044 -> 456 us each, clearing 179 -> 135 us a tree, the fit 18.0 -> 16.3 ms.
  const bool plain = observes_nothing(taps);
  bool lazy = false, strict = false;
  bool kept        = false;  // the level before left its scanned histograms in the buffer
  int cleared_end  = hv.node_end;
  if (plain) {
    constexpr uint64_t kAtOnce = 64 << 20;
    int first = 0;
    while (first + 1 <= max_depth && level_end(first + 1) <= hv.node_end &&
           static_cast<uint64_t>(level_end(first + 1)) * bytes_per_node <= kAtOnce)
      first++;
    cleared_end = std::min(hv.node_end, static_cast<int>(level_end(first)));
  }
  RootArgs root{leaf, L.node_sums, K, L.scales, prm.l1_regularization, prm.l2_regularization, L.qstats, reinterpret_cast<unsigned long long*>(hm->mirror), nullptr, 0};
  LBT_TRY(hist_range(hv.node_begin, cleared_end, &root.clear, &root.n16));
  LBT_TRY(hist_prepare(stream, hs, sizeof(T) == 8, F, K, N, rp, L.proposals, L.row_pointers, X, &root));
  LBT_HIP(hipEventRecord(hm->stats_here, stream));
  //  - Single-output trees: levels whose histograms are larger than the rows' records keep them in the LDS
  //    (1,000,000 x 50 with 512 samples: level 11 743 -> 176 us, level 10 356 -> 108, level 9, the first with larger
  //    ones, 193 -> 92; with level 8, whose histograms are 0.8 of the records, a balanced tree would take 1.56 ms instead of
  //    1.62, one of noise, whose large nodes are added range by range, 2.07 instead of 1.97).
  int direct_from = max_depth;
  int range_of_large = 0;   // of a direct level
  bool large_ready = false;  // the histograms of large nodes lie where other levels' did, and begin at zero
  if (plain && L.left != nullptr && hs.binned != nullptr && hs.embed && hs.max_bins <= kDirectMaxBins &&
      N < (int64_t(1) << 30) && (range_of_large = direct_range(hs, N, L.hist_bytes)) > 0) {
    direct_from = 2;  // at the root it is not known yet
    while (direct_from < max_depth && static_cast<double>(bytes_per_node) * static_cast<double>(int64_t(1) << direct_from) <
                                        static_cast<double>(N) * static_cast<double>(hs.row_bytes))
      direct_from++;
  }
  int cur_pos = 0, cur_seg = 0;
  // the feature-major bins serve the position updates of levels 0 .. max_depth-2
  const bool use_bins_t = hs.binned != nullptr && L.bins_t != nullptr;
  int32_t* row_leaf     = taps ? taps->row_leaf : nullptr;
  const int n_chunks = (B + kSplitChunk - 1) / kSplitChunk;
  ScatterArgs scatter{};
  bool scatter_due = false;
  auto scatter_now = [&]() {
    if (!scatter_due) return;
    ProfScope ps(LBT_PROF_POSITIONS, stream, static_cast<double>(N) * (4 + 1 + 4));
    scatter_kernel<<<blocks(N, kPartBlock), kThreads, 0, stream>>>(scatter);
    scatter_due = false;
  };
  for (int depth = 0; depth < max_depth; depth++) {
    const int64_t nodes_in_level = int64_t(1) << depth;
    const int level_first        = static_cast<int>(level_begin(depth));
    if (taps && taps->positions_per_level) {
      scatter_now();
      expand_positions_kernel<<<blocks(N, kPartBlock), kThreads, 0, stream>>>(
        L.rows[cur_pos], N, L.seg[cur_seg], L.block_seg[cur_seg], static_cast<int>(nodes_in_level), level_first,
        reinterpret_cast<int2*>(taps->positions_per_level) + static_cast<size_t>(depth) * N);
    }
    int clear_from = 0, clear_nodes = 0, clear_parts = 1;  // built histograms of the level to clear
    const bool direct = lazy && depth >= direct_from;
    if (lazy && !direct) {
      const int64_t end = level_end(depth);
      if (end > hv.node_end && kept && prm.hist_cache_bytes == 0 && hv.node_begin == 0 &&
          static_cast<uint64_t>(end) * bytes_per_node <= L.hist_bytes) {
        hv.node_end = static_cast<int>(end);
        if (strict) hv.tainted = L.tainted;
      }
      if (end <= hv.node_end && hv.node_begin == 0 && end > cleared_end) {
        clear_from  = std::max(cleared_end, level_first);
        clear_nodes = static_cast<int>(end) - clear_from;
        clear_parts = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(static_cast<int64_t>(K) * B / (4 * kThreads), 64)));
        cleared_end = static_cast<int>(end);
      }
    }
    uint8_t* const taint = strict && hv.tainted == nullptr ? L.tainted : nullptr;
    const bool contained         = level_first >= hv.node_begin && level_end(depth) <= hv.node_end;
    int64_t num_batches          = 1;
    if (nodes_in_level > max_batch_size && !(lazy && contained)) num_batches = (nodes_in_level + max_batch_size - 1) / max_batch_size;
    auto batch_of = [&](int j0, int j1) {
      HistBatch hb;
      hb.X = X; hb.F = F; hb.qgh = L.qgh; hb.K = K; hb.rows = L.rows[cur_pos]; hb.seg = L.seg[cur_seg];
      hb.j0 = j0; hb.n_nodes = j1 - j0; hb.level_first = level_first; hb.proposals = L.proposals;
      hb.row_pointers = L.row_pointers; hb.bin_feature = L.bin_feature; hb.hist = hv; hb.qstats = L.qstats; hb.node_sums = L.node_sums;
      hb.level_total = L.level_totals + depth; hb.n_rows = N;
      // the root's rows are still in their original order, and its launch fills the bin cache first
      hb.fill_cache = depth == 0; hb.identity = depth == 0;
      return hb;
    };
    bool planned = false, decides = false;  // decides: the level's splits are applied where its rows are classified
    DecideArgs decide{};
    if (scatter_due && !direct && num_batches == 1 && contained) {
      PlanArgs plan;
      LBT_TRY(hist_plan(hs, batch_of(0, static_cast<int>(nodes_in_level)), &plan));
      if (plan.blocks > 0) {
        ProfScope ps(LBT_PROF_POSITIONS, stream, static_cast<double>(N) * (4 + 1 + 4));
        const unsigned nb = blocks(N, kPartBlock);
        level_start_kernel<<<(plan.blocks + 7) / 8 * 8 + nb + clear_nodes * clear_parts, kThreads, 0, stream>>>(plan, scatter, static_cast<int>(nb), clear_from,
                                                                                                 clear_parts);
        scatter_due = false;
        clear_nodes = 0;
        planned     = true;
      }
    }
    scatter_now();
    if (clear_nodes > 0)
      zero_built_kernel<<<dim3(clear_nodes, clear_parts), kThreads, 0, stream>>>(hv, L.node_sums, clear_from);
    if (direct) {
      const int64_t large16 = static_cast<int64_t>(direct_large_bytes(hs, N, range_of_large) / 16);
      if (!large_ready && large16 > 0) {
        ProfScope ps(LBT_PROF_OTHER, stream, 16.0 * static_cast<double>(large16));
        zero_kernel<<<static_cast<unsigned>(std::min<int64_t>((large16 + kThreads - 1) / kThreads, 65536)), kThreads, 0, stream>>>(
          reinterpret_cast<uint4*>(L.hist), large16);
      }
      large_ready = true;
      DirectLevel dl;
      dl.level_first = level_first; dl.n_nodes = static_cast<int>(nodes_in_level); dl.n_features = F;
      dl.n_groups = hs.n_groups; dl.n_rows = N; dl.binned = hs.binned; dl.rec = hs.rec; dl.groups = hs.groups;
      dl.block_seg = L.block_seg[cur_seg]; dl.slab = kPartBlock; dl.range = range_of_large; dl.large = reinterpret_cast<unsigned long long*>(L.hist);
      dl.arrivals = nullptr;
      dl.rows = L.rows[cur_pos]; dl.seg = L.seg[cur_seg]; dl.row_pointers = L.row_pointers; dl.feature_set = feature_set;
      dl.scales = L.scales; dl.l1 = prm.l1_regularization; dl.l2 = prm.l2_regularization;
      dl.min_split_gain = prm.min_split_gain; dl.proposals = L.proposals_d; dl.node_sums = L.node_sums;
      dl.partial = L.partial; dl.left = L.left; dl.leaf = leaf; dl.feature = feature; dl.split = split; dl.gain = gain;
      dl.split_bin = L.split_bin;
      LBT_TRY(direct_level_launch(stream, dl, hs));
      num_batches = 0;
    }
    for (int64_t bi = 0; bi < num_batches; bi++) {
      int j0 = 0, j1 = static_cast<int>(nodes_in_level);
      if (num_batches > 1) {
        j0 = static_cast<int>(bi * max_batch_size);
        j1 = static_cast<int>(std::min<int64_t>(j0 + max_batch_size, nodes_in_level));
      }
      const int batch_begin = level_first + j0, batch_end = level_first + j1;
      // GetHistogram (build_tree.cu:1191-1205)
      if (!(batch_begin >= hv.node_begin && batch_end <= hv.node_end)) {
        hv.node_begin = batch_begin;
        hv.node_end   = batch_end;
        hv.tainted    = nullptr;
        cleared_end   = batch_end;
        LBT_TRY(zero_hist(hv.node_begin, hv.node_end));
      }
      const int n_nodes = j1 - j0;
      {
        HistBatch hb = batch_of(j0, j1);
        hb.planned   = planned;
        LBT_TRY(hist_launch(stream, hs, hb, depth));
      }
      // One pass that scans and evaluates reads the histograms once instead of twice and saves a
      // launch per level. With a single output and many nodes (the deep levels of a deep tree,
      // most of whose nodes are empty or small) the two kernels are faster: the evaluation then
      // runs over all bins of a node side by side, not feature by feature behind the scan.
      // The scanned histograms of this level are read again only by the next level's sibling
      // subtraction (and by a caller that asked to see them): not after the last level, and not
      // when the next level starts a buffer of its own (GetHistogram, build_tree.cu:1191-1205).
      const int64_t next_begin = level_begin(depth + 1), next_end = level_end(depth + 1);
      const bool next_grows    = lazy && prm.hist_cache_bytes == 0 && hv.node_begin == 0 &&
                              static_cast<uint64_t>(next_end) * bytes_per_node <= L.hist_bytes;
      const bool next_reads    = depth + 1 < max_depth && !(lazy && depth + 1 >= direct_from) &&
                              (next_grows || (next_end - next_begin <= max_batch_size &&
                                              next_begin >= hv.node_begin && next_end <= hv.node_end));
      const bool wanted = next_reads || (taps && taps->histogram);
      // ... and where nothing reads them again the fused pass, which then only reads, wins as well
      const bool fused = narrow_sums_hold(N) && K <= kFusedMaxK && (K >= 2 || n_nodes <= 256 || !wanted);
      const bool store = !fused || wanted;
      kept             = store;
      const int n_cands = fused ? F : n_chunks;
      // (with negative hessians a node without rows may have a split)
      decides = N <= kDecideRows && (depth == 0 || lazy) && depth < max_depth - 1 && use_bins_t && num_batches == 1 && store &&
                n_cands <= kDecideCands && K <= 64 && nodes_in_level <= kDecideNodes;
      if (fused) {
        ProfScope ps(LBT_PROF_SCAN, stream);
        scan_split_launch(stream, hs.max_bins, hv, L.node_sums, F, L.row_pointers, batch_begin, n_nodes, feature_set,
                          L.scales, prm.l1_regularization, prm.l2_regularization, prm.min_split_gain, L.partial, N, store, taint);
      } else {
        {
          ProfScope ps(LBT_PROF_SCAN, stream);
          int64_t waves = static_cast<int64_t>(F) * n_nodes;
          dim3 grid(blocks(waves, kThreads / 64), K);
          scan_kernel<<<grid, kThreads, 0, stream>>>(hv, L.node_sums, F, L.row_pointers, batch_begin, n_nodes, taint);
        }
        ProfScope ps(LBT_PROF_SPLIT, stream);
        dim3 grid(n_nodes, n_chunks);
        split_eval_kernel<<<grid, kThreads, 0, stream>>>(hv, L.node_sums, L.bin_feature, feature_set, L.scales,
                                                         prm.l1_regularization, prm.l2_regularization,
                                                         prm.min_split_gain, batch_begin, n_chunks, L.partial);
      }
      if (decides) {
        decide = DecideArgs{hv, L.node_sums, L.bin_feature, L.proposals_d, L.scales, prm.l1_regularization, prm.l2_regularization, n_cands,
                            L.partial, leaf, feature, split, gain, L.row_pointers, L.split_bin};
      } else {
        ProfScope ps(LBT_PROF_SPLIT, stream);
        split_apply_kernel<<<n_nodes, 64, 0, stream>>>(hv, L.node_sums, L.bin_feature, L.proposals_d, L.scales,
                                                       prm.l1_regularization, prm.l2_regularization, batch_begin,
                                                       n_cands, L.partial, leaf, feature, split, gain, L.row_pointers,
                                                       L.split_bin, store);
      }
    }
    if (depth < max_depth - 1) {
      ProfScope ps(LBT_PROF_POSITIONS, stream, static_cast<double>(N) * (4 + 4 + 2 + 64));
      const unsigned nb   = blocks(N, kPartBlock);
      const int n_parents = static_cast<int>(nodes_in_level);
      const int32_t* rows = L.rows[cur_pos];
      const int32_t* seg  = L.seg[cur_seg];
      const int32_t* bseg = L.block_seg[cur_seg];
      auto classify_bins = [&](auto kernel, const auto* bins) {
        kernel<<<nb, kThreads, 0, stream>>>(rows, N, seg, bseg, n_parents, level_first, bins, L.bins_t_stride, feature,
                                            L.split_bin, L.code, L.block_counts, decide);
      };
      const bool runs = classify_in_runs(n_parents, N);
      auto classify_as = [&](auto bin, auto decides_c) {
        using BinT          = decltype(bin);
        constexpr bool kDec = decltype(decides_c)::value;
        classify_bins(runs ? classify_bins_kernel<BinT, true, kDec> : classify_bins_kernel<BinT, false, kDec>,
                      static_cast<const BinT*>(L.bins_t));
      };
      auto classify_of = [&](auto bin) { decides ? classify_as(bin, std::true_type{}) : classify_as(bin, std::false_type{}); };
      if (use_bins_t && hs.bin_bytes == 1)
        classify_of(uint8_t{});
      else if (use_bins_t)
        classify_of(uint16_t{});
      else
        classify_kernel<T><<<nb, kThreads, 0, stream>>>(rows, N, seg, bseg, n_parents, level_first, X, F, feature, split,
                                                        L.code, L.block_counts);
      child_segments_kernel<<<blocks(n_parents, kScanThreads / 64), kScanThreads, 0, stream>>>(
        seg, n_parents, N, L.code, L.block_counts, static_cast<int>(nb), L.block_offsets, L.seg_prefix,
        L.seg[cur_seg ^ 1], L.block_seg[cur_seg ^ 1]);
      scatter = ScatterArgs{rows, N, L.code, L.block_offsets, seg, bseg, L.seg_prefix, L.seg[cur_seg ^ 1], level_first, n_parents,
                            L.rows[cur_pos ^ 1], row_leaf};
      scatter_due = true;  // with what the next level begins with
      cur_pos ^= 1;
      cur_seg ^= 1;
    }
    if (depth == 0) {
      LBT_TRY(check_stats());
      lazy   = plain && (h_qstats[1] & kQuantHessNegative) == 0;
      strict = lazy && (h_qstats[1] & kQuantHessNotPositive) != 0;
      if (strict) direct_from = max_depth;  // (their nodes are added up from their rows)
      if (!lazy && cleared_end < hv.node_end) LBT_TRY(zero_hist(cleared_end, hv.node_end));
    }
  }
  LBT_TRY(check_stats());

  if (row_leaf != nullptr) {
    ProfScope ps(LBT_PROF_POSITIONS, stream);
    const bool bt = use_bins_t && max_depth >= 2;
    const int n_parents = static_cast<int>(int64_t(1) << (max_depth > 0 ? max_depth - 1 : 0));
    const int n_windows = static_cast<int>((N + kLeafWindow - 1) / kLeafWindow);
    const int64_t bound_entries = static_cast<int64_t>(n_parents) * (n_windows + 1);
    // the order of the last level: segments level_first .. level_first + n_parents - 1
    const int level_first = static_cast<int>(level_begin(max_depth > 0 ? max_depth - 1 : 0));
    if (bt && n_parents <= kLeafParents && bound_entries <= kLeafBoundsEntries) {
      leaf_window_bounds_kernel<<<blocks(bound_entries, kThreads), kThreads, 0, stream>>>(
        L.rows[cur_pos], L.seg[cur_seg], n_parents, n_windows, L.leaf_bounds);
      if (hs.bin_bytes == 2)
        final_leaf_window_kernel<uint16_t><<<n_windows, kLeafThreads, 0, stream>>>(
          L.rows[cur_pos], L.leaf_bounds, n_parents, n_windows, level_first, static_cast<const uint16_t*>(L.bins_t),
          L.bins_t_stride, feature, L.split_bin, row_leaf);
      else
        final_leaf_window_kernel<uint8_t><<<n_windows, kLeafThreads, 0, stream>>>(
          L.rows[cur_pos], L.leaf_bounds, n_parents, n_windows, level_first, static_cast<const uint8_t*>(L.bins_t),
          L.bins_t_stride, feature, L.split_bin, row_leaf);
    } else if (bt && hs.bin_bytes == 2)
      final_leaf_kernel<T, uint16_t><<<blocks(N, kPartBlock), kThreads, 0, stream>>>(
        L.rows[cur_pos], N, L.seg[cur_seg], L.block_seg[cur_seg], n_parents, level_first, X, F,
        static_cast<const uint16_t*>(L.bins_t), L.bins_t_stride, feature, split, L.split_bin, row_leaf);
    else
      final_leaf_kernel<T, uint8_t><<<blocks(N, kPartBlock), kThreads, 0, stream>>>(
        L.rows[cur_pos], N, L.seg[cur_seg], L.block_seg[cur_seg], n_parents, level_first, X, F,
        bt ? static_cast<const uint8_t*>(L.bins_t) : nullptr, L.bins_t_stride, feature, split, L.split_bin, row_leaf);
  }
  {
    ProfScope ps(LBT_PROF_OTHER, stream);
    write_hessian_kernel<<<blocks(static_cast<int64_t>(max_nodes) * K, kThreads), kThreads, 0, stream>>>(
      hessian, L.node_sums, static_cast<int64_t>(max_nodes) * K, L.scales);
  }

  // ---- observation points
  const bool tap_levels =
    taps && (taps->level_instances || taps->level_built_instances || taps->level_built_nodes) && max_depth > 0;
  if (profiler().mode != 0 && max_depth > 0) {
    // bytes of one feature value as the level reads it (X itself, or its cached bin)
    const bool cached      = hs.binned != nullptr;
    const double per_value = cached ? hs.bin_bytes : static_cast<double>(sizeof(T));
    LBT_TRY(profile_levels(stream, L.level_totals, max_depth, static_cast<double>(F) * per_value + K * 8.0 + 8.0,
                           static_cast<double>(K) * B * 16.0,
                           // the root launch also writes the feature-major copy of the bins
                           hs.bins_t != nullptr ? static_cast<double>(N) * F * hs.bin_bytes : 0.0));
  }
  std::vector<LevelMeta> h_levels(max_depth > 0 ? max_depth : 1);
  if (tap_levels && sync_at_end)
    LBT_HIP(hipMemcpyAsync(h_levels.data(), L.level_totals, sizeof(LevelMeta) * max_depth, hipMemcpyDeviceToHost, stream));
  if (taps) {
    taps->n_bins          = B;
    taps->hist_node_begin = hv.node_begin;
    taps->hist_node_end   = static_cast<int32_t>(std::max<int64_t>(hv.node_begin, std::min<int64_t>(hv.node_end, used_end)));
    // host members that come from the device are filled only by the call that waits for them
    if (sync_at_end) LBT_HIP(hipMemcpyAsync(taps->scales, L.scales, sizeof(double) * 4, hipMemcpyDeviceToHost, stream));
    if (taps->proposals)
      LBT_HIP(hipMemcpyAsync(taps->proposals, L.proposals, sizeof(T) * B, hipMemcpyDeviceToDevice, stream));
    if (taps->row_pointers)
      LBT_HIP(hipMemcpyAsync(taps->row_pointers, L.row_pointers, sizeof(int32_t) * (F + 1), hipMemcpyDeviceToDevice, stream));
    if (taps->quantised)
      LBT_HIP(hipMemcpyAsync(taps->quantised, L.qgh, sizeof(int2) * N * K, hipMemcpyDeviceToDevice, stream));
    if (taps->node_sums)
      LBT_HIP(hipMemcpyAsync(taps->node_sums, L.node_sums, sizeof(I64Pair) * max_nodes * K, hipMemcpyDeviceToDevice, stream));
    if (taps->positions) {
      const int last = max_depth > 0 ? max_depth - 1 : 0;
      expand_positions_kernel<<<blocks(N, kPartBlock), kThreads, 0, stream>>>(
        L.rows[cur_pos], N, L.seg[cur_seg], L.block_seg[cur_seg], static_cast<int>(int64_t(1) << last),
        static_cast<int>(level_begin(last)), reinterpret_cast<int2*>(taps->positions));
    }
    if (taps->histogram) {
      int64_t nodes = taps->hist_node_end - taps->hist_node_begin;
      int64_t need  = nodes * K * B * 2;
      if (need > 0 && need <= taps->histogram_capacity)
        LBT_HIP(hipMemcpyAsync(taps->histogram, L.hist, sizeof(int64_t) * need, hipMemcpyDeviceToDevice, stream));
    }
  }
  LBT_HIP(hipGetLastError());
  if (!sync_at_end) return LBT_OK;
  LBT_HIP(hipStreamSynchronize(stream));
  LBT_HIP(hipGetLastError());
  if (tap_levels) {
    for (int d = 0; d < max_depth; d++) {
      if (taps->level_instances) taps->level_instances[d] = h_levels[d].instances;
      if (taps->level_built_instances) taps->level_built_instances[d] = h_levels[d].built_instances;
      if (taps->level_built_nodes) taps->level_built_nodes[d] = static_cast<int32_t>(h_levels[d].built_nodes);
    }
  }
  if (profiler().mode != 0) profiler().collect();
  return LBT_OK;
}

}  // namespace
}  // namespace lbt

namespace {

struct SampleScratch {
  char* uniq;
  int32_t* counts;
  int32_t* bin_feature;
};
void make_sample_scratch(lbt::Arena& ar, SampleScratch& w, int F, int S, size_t elem)
{
  w.uniq        = ar.take<char>(static_cast<size_t>(F) * S * elem);
  w.counts      = ar.take<int32_t>(F);
  w.bin_feature = ar.take<int32_t>(static_cast<size_t>(F) * S);
}

struct QuantiserScratch {
  double* part_a[2];
  double* part_b[2];
  unsigned long long* qstats;
};
void make_quantiser_scratch(lbt::Arena& ar, QuantiserScratch& w, int64_t N, int K)
{
  int64_t n_chunks = (N * K + 4095) / 4096;
  for (int i = 0; i < 2; i++) {
    w.part_a[i] = ar.take<double>(n_chunks);
    w.part_b[i] = ar.take<double>(n_chunks);
    n_chunks    = (n_chunks + 4095) / 4096;
  }
  w.qstats = ar.take<unsigned long long>(2);
}

int arena_over(lbt::Arena& ar, void* workspace, size_t workspace_bytes)
{
  if (workspace == nullptr) {
    lbt::set_error("workspace is null");
    return LBT_ERR_WORKSPACE;
  }
  const uintptr_t raw     = reinterpret_cast<uintptr_t>(workspace);
  const uintptr_t aligned = (raw + 255) & ~uintptr_t(255);
  ar.base                 = reinterpret_cast<char*>(aligned);
  ar.cap                  = workspace_bytes > (aligned - raw) ? workspace_bytes - (aligned - raw) : 0;
  return LBT_OK;
}

}  // namespace

extern "C" {

size_t lbt_build_tree_workspace_bytes(int64_t n_rows, int32_t n_features, int32_t n_outputs,
                                      int32_t max_depth, int32_t split_samples, int32_t x_dtype,
                                      int64_t hist_cache_bytes)
{
  lbt_build_params p{};
  p.struct_bytes     = static_cast<int32_t>(sizeof(p));
  p.max_depth        = max_depth;
  p.max_nodes        = max_depth >= 0 && max_depth <= 24 ? static_cast<int32_t>(lbt::level_end(max_depth)) : 0;
  p.split_samples    = split_samples;
  p.dataset_rows     = 1;
  p.hist_cache_bytes = hist_cache_bytes;
  if (lbt::validate(n_rows, n_features, n_outputs, &p, x_dtype) != LBT_OK) return 0;
  lbt::Arena ar;
  ar.measure = true;
  lbt::Layout L{};
  lbt::make_layout(ar, L, n_rows, n_features, n_outputs, max_depth, split_samples,
                   x_dtype == LBT_F64 ? 8 : 4, hist_cache_bytes, true);
  return ar.used + 256;
}

static int build_tree_entry(void* stream, const void* X, int32_t x_dtype, int64_t row_offset, int64_t n_rows,
                            int32_t n_features, const double* g, const double* h, int32_t n_outputs,
                            const uint8_t* feature_set, const lbt_build_params* params, double* leaf, int32_t* feature,
                            double* split, double* gain, double* hessian, void* workspace, size_t workspace_bytes,
                            lbt_build_taps* taps, bool sync_at_end)
{
  LBT_TRY(lbt::validate(n_rows, n_features, n_outputs, params, x_dtype));
  LBT_REQUIRE(X && g && h && leaf && feature && split && gain && hessian, "null input or output pointer");
  LBT_REQUIRE(row_offset >= 0, "row_offset must not be negative");
  if (params->abs_sum_chunks != nullptr) {
    // the chunk sums are read while g and h may still be in use by the same pass: no overlap
    const char* c0 = reinterpret_cast<const char*>(params->abs_sum_chunks);
    const char* c1 = c0 + 2 * sizeof(double) * static_cast<size_t>((n_rows * n_outputs + 4095) / 4096);
    const size_t gh_bytes = sizeof(double) * static_cast<size_t>(n_rows) * n_outputs;
    for (const double* a : {g, h}) {
      const char* a0 = reinterpret_cast<const char*>(a);
      LBT_REQUIRE(c1 <= a0 || a0 + gh_bytes <= c0, "abs_sum_chunks overlaps g or h");
    }
  }
  if (workspace == nullptr) {
    lbt::set_error("workspace is null; size it with lbt_build_tree_workspace_bytes");
    return LBT_ERR_WORKSPACE;
  }
  lbt::Arena ar;
  uintptr_t raw     = reinterpret_cast<uintptr_t>(workspace);
  uintptr_t aligned = (raw + 255) & ~uintptr_t(255);
  ar.base           = reinterpret_cast<char*>(aligned);
  ar.cap            = workspace_bytes > (aligned - raw) ? workspace_bytes - (aligned - raw) : 0;
  const lbt::Arena whole = ar;
  lbt::Layout L{};
  for (const bool roomy : {true, false}) {  // a workspace that holds the reference's budget only is enough
    ar = whole;
    L  = lbt::Layout{};
    lbt::make_layout(ar, L, n_rows, n_features, n_outputs, params->max_depth, params->split_samples,
                     x_dtype == LBT_F64 ? 8 : 4, params->hist_cache_bytes, roomy);
    if (!ar.failed) break;
  }
  if (ar.failed) {
    lbt::set_error("workspace too small: %zu bytes given, %zu needed", workspace_bytes, ar.used + 256);
    return LBT_ERR_WORKSPACE;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  int rc        = LBT_OK;
  bool done     = false;
  // the builders for few rows and medium sizes, unless the caller wants to see what they do not have
  if (lbt::observes_nothing(taps) && (L.small.order[0] != nullptr || L.mid.bins != nullptr)) {
    int32_t* const row_leaf = taps ? taps->row_leaf : nullptr;
    int32_t* const n_bins   = taps ? &taps->n_bins : nullptr;
    const float* const Xf   = static_cast<const float*>(X);
    const double* const Xd  = static_cast<const double*>(X);
    lbt::LevelMeta* totals  = nullptr;
    if (lbt::profiler().mode != 0) {
      totals = L.level_totals;
      lbt::zero_kernel<<<1, lbt::kThreads, 0, s>>>(reinterpret_cast<uint4*>(totals), 2 * params->max_depth);
    }
    if (L.small.order[0] != nullptr)
      rc = x_dtype == LBT_F32
             ? lbt::small_tree_build<float>(s, L.small, Xf, row_offset, n_rows, n_features, n_outputs, g, h, feature_set,
                                            *params, leaf, feature, split, gain, hessian, row_leaf, n_bins, totals, &done)
             : lbt::small_tree_build<double>(s, L.small, Xd, row_offset, n_rows, n_features, n_outputs, g, h, feature_set,
                                             *params, leaf, feature, split, gain, hessian, row_leaf, n_bins, totals, &done);
    else
      rc = x_dtype == LBT_F32
             ? lbt::mid_tree_build<float>(s, L.mid, Xf, row_offset, n_rows, n_features, n_outputs, g, h, feature_set,
                                          *params, leaf, feature, split, gain, hessian, row_leaf, n_bins, totals, &done)
             : lbt::mid_tree_build<double>(s, L.mid, Xd, row_offset, n_rows, n_features, n_outputs, g, h, feature_set,
                                           *params, leaf, feature, split, gain, hessian, row_leaf, n_bins, totals, &done);
    if (rc == LBT_OK && done) {
      if (taps) {
        lbt::final_histogram_range(n_outputs, taps->n_bins, *params, &taps->hist_node_begin, &taps->hist_node_end);
        if (sync_at_end) LBT_HIP(hipMemcpyAsync(taps->scales, L.scales, sizeof(double) * 4, hipMemcpyDeviceToHost, s));
      }
      if (totals != nullptr) {
        const double row_bytes = static_cast<double>(n_features) * (params->split_samples <= 256 ? 1 : 2) + n_outputs * 8.0 + 8.0;
        LBT_TRY(lbt::profile_levels(s, L.level_totals, params->max_depth, row_bytes,
                                    static_cast<double>(n_outputs) * n_features * params->split_samples * 16.0, 0.0));
      }
      if (!sync_at_end) return LBT_OK;
      LBT_HIP(hipStreamSynchronize(s));
      LBT_HIP(hipGetLastError());
      if (lbt::profiler().mode != 0) lbt::profiler().collect();
      return LBT_OK;
    }
  }
  if (rc != LBT_OK) {
  } else if (x_dtype == LBT_F32)
    rc = lbt::build_tree_impl<float>(s, static_cast<const float*>(X), row_offset, n_rows, n_features, g, h, n_outputs,
                                     feature_set, *params, leaf, feature, split, gain, hessian, L, taps, sync_at_end);
  else
    rc = lbt::build_tree_impl<double>(s, static_cast<const double*>(X), row_offset, n_rows, n_features, g, h, n_outputs,
                                      feature_set, *params, leaf, feature, split, gain, hessian, L, taps, sync_at_end);
  if (rc != LBT_OK) {
    // Kernels of the stages before the failure may still be queued and write to the outputs and
    // the workspace. The synchronising entry drains them, so that the caller may release both as
    // soon as it sees the status (the task glue throws, and Legate then frees the buffers); the
    // message of the failure is kept. The asynchronous entry leaves the wait to its caller.
    if (sync_at_end || lbt::profiler().mode != 0) (void)hipStreamSynchronize(s);
    if (lbt::profiler().mode != 0) lbt::profiler().collect();
  }
  return rc;
}

size_t lbt_select_split_samples_workspace_bytes(int32_t n_features, int32_t split_samples, int32_t x_dtype)
{
  if (n_features < 1 || split_samples < 1 || split_samples > LBT_MAX_SPLIT_SAMPLES) return 0;
  if (x_dtype != LBT_F32 && x_dtype != LBT_F64) return 0;
  lbt::Arena ar;
  ar.measure = true;
  SampleScratch w;
  make_sample_scratch(ar, w, n_features, split_samples, x_dtype == LBT_F64 ? 8 : 4);
  return ar.used + 256;
}

int lbt_select_split_samples(void* stream, const void* X, int32_t x_dtype, int64_t row_offset, int64_t n_rows,
                             int32_t n_features, int32_t split_samples, int32_t seed, int64_t dataset_rows,
                             void* proposals, int32_t* row_pointers, void* workspace, size_t workspace_bytes)
{
  LBT_REQUIRE(x_dtype == LBT_F32 || x_dtype == LBT_F64, "unsupported X dtype %d", x_dtype);
  LBT_REQUIRE(n_rows >= 0 && n_rows < 2147483647LL && n_features >= 1, "bad shape");
  LBT_REQUIRE(split_samples >= 1 && split_samples <= LBT_MAX_SPLIT_SAMPLES, "split_samples must be in [1, %d]",
              LBT_MAX_SPLIT_SAMPLES);
  LBT_REQUIRE(dataset_rows >= 1 && row_offset >= 0, "dataset_rows must be positive, row_offset not negative");
  LBT_REQUIRE((X || n_rows == 0) && proposals && row_pointers, "null input or output pointer");
  lbt::Arena ar;
  LBT_TRY(arena_over(ar, workspace, workspace_bytes));
  SampleScratch w;
  make_sample_scratch(ar, w, n_features, split_samples, x_dtype == LBT_F64 ? 8 : 4);
  if (ar.failed) {
    lbt::set_error("workspace too small: %zu bytes given, %zu needed", workspace_bytes, ar.used + 256);
    return LBT_ERR_WORKSPACE;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  lbt::ProfScope ps(LBT_PROF_PROPOSALS, s);
  auto run = [&](auto type) {
    using T = decltype(type);
    return lbt::run_split_samples<T>(s, lbt::SampleArgs<T>{static_cast<const T*>(X), row_offset, n_rows, dataset_rows, n_features, split_samples, 0, seed,
                                                           reinterpret_cast<T*>(w.uniq), w.counts, row_pointers, static_cast<T*>(proposals), w.bin_feature,
                                                           nullptr, nullptr});
  };
  return x_dtype == LBT_F32 ? run(float{}) : run(double{});
}

size_t lbt_quantise_gradients_workspace_bytes(int64_t n_rows, int32_t n_outputs)
{
  if (n_rows < 1 || n_outputs < 1 || n_rows >= 2147483647LL) return 0;
  lbt::Arena ar;
  ar.measure = true;
  QuantiserScratch w;
  make_quantiser_scratch(ar, w, n_rows, n_outputs);
  return ar.used + 256;
}

int lbt_quantise_gradients(void* stream, const double* g, const double* h, int64_t n_rows, int32_t n_outputs,
                           int64_t row_offset, int32_t seed, int32_t* quantised, int64_t* root_sums, double* scales,
                           void* workspace, size_t workspace_bytes)
{
  LBT_REQUIRE(n_rows >= 1 && n_rows < 2147483647LL && n_outputs >= 1 && n_outputs <= 65535, "bad shape");
  LBT_REQUIRE(row_offset >= 0, "row_offset must not be negative");
  LBT_REQUIRE(g && h && quantised && root_sums && scales, "null input or output pointer");
  LBT_REQUIRE(reinterpret_cast<uintptr_t>(root_sums) % 16 == 0, "root_sums must be 16-byte aligned");
  lbt::Arena ar;
  LBT_TRY(arena_over(ar, workspace, workspace_bytes));
  QuantiserScratch w;
  make_quantiser_scratch(ar, w, n_rows, n_outputs);
  if (ar.failed) {
    lbt::set_error("workspace too small: %zu bytes given, %zu needed", workspace_bytes, ar.used + 256);
    return LBT_ERR_WORKSPACE;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  lbt::ProfScope ps(LBT_PROF_QUANTISE, s, static_cast<double>(n_rows) * n_outputs * (16 + 16 + 8));
  // the sums are added to: clear them with a kernel (a memset node would not replay in a captured graph)
  static_assert(sizeof(lbt::I64Pair) == 16, "root sums are cleared in 16-byte units");
  lbt::zero_kernel<<<1, lbt::kThreads, 0, s>>>(reinterpret_cast<uint4*>(root_sums), n_outputs);
  return lbt::run_quantiser(s, g, h, n_rows, n_outputs, row_offset, seed, w.part_a, w.part_b, scales, w.qstats,
                            reinterpret_cast<int2*>(quantised), reinterpret_cast<lbt::I64Pair*>(root_sums));
}

}  // extern "C"

// ---------------------------------------------------------------------------
// The quantiser for callers that cannot allocate: its scratch (the partial sums of the two
// absolute sums and the two statistics words) lives in a device array of this library instead
// of a caller's workspace. Every GPU the library is loaded on holds its own copy of the array
// until the process ends. `static_scratch` is only the host-side handle of it: what kernels and
// copies are given is the address that hipGetSymbolAddress returns for the current device.
// ---------------------------------------------------------------------------
namespace {

constexpr int64_t kStaticMaxEntries = LBT_QUANTISE_STATIC_MAX_ENTRIES;  // n_rows * n_outputs
// two levels of partial sums (one double per 4096 entries, twice) for g and h, 256-byte pitch, and qstats
constexpr size_t kStaticScratchBytes =
  2 * (((static_cast<size_t>(kStaticMaxEntries) / 4096 * sizeof(double)) + 255) / 256 * 256) + 2 * 256 + 256 + 256;
static __device__ __align__(256) unsigned char static_scratch[kStaticScratchBytes];

std::atomic<void*> static_scratch_ptr[lbt::kMaxDevices] = {};

// The array's address on the current device, resolved once per device.
int static_scratch_address(void** out)
{
  int device = 0;
  LBT_HIP(hipGetDevice(&device));
  LBT_REQUIRE(device >= 0 && device < lbt::kMaxDevices, "device ordinal %d is not supported", device);
  void* p = static_scratch_ptr[device].load(std::memory_order_acquire);
  if (p == nullptr) {
    LBT_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(static_scratch)));
    LBT_REQUIRE(p != nullptr, "the address of the static scratch array is null");
    static_scratch_ptr[device].store(p, std::memory_order_release);  // two threads resolve the same address
  }
  *out = p;
  return LBT_OK;
}

}  // namespace

extern "C" {

int lbt_quantise_gradients_static(void* stream, const double* g, const double* h, int64_t n_rows, int32_t n_outputs,
                                  int64_t row_offset, int32_t seed, int32_t* quantised, int64_t* root_sums,
                                  double* scales)
{
  LBT_REQUIRE(n_rows >= 1 && n_rows < 2147483647LL && n_outputs >= 1 && n_outputs <= 65535, "bad shape");
  LBT_REQUIRE(n_rows * static_cast<int64_t>(n_outputs) <= kStaticMaxEntries,
              "lbt_quantise_gradients_static takes at most %lld entries (n_rows * n_outputs), got %lld: use "
              "lbt_quantise_gradients with a workspace",
              static_cast<long long>(kStaticMaxEntries), static_cast<long long>(n_rows * static_cast<int64_t>(n_outputs)));
  LBT_REQUIRE(row_offset >= 0, "row_offset must not be negative");
  LBT_REQUIRE(g && h && quantised && root_sums && scales, "null input or output pointer");
  LBT_REQUIRE(reinterpret_cast<uintptr_t>(root_sums) % 16 == 0, "root_sums must be 16-byte aligned");
  void* scratch = nullptr;
  LBT_TRY(static_scratch_address(&scratch));
  lbt::Arena ar;
  ar.base = static_cast<char*>(scratch);
  ar.cap  = kStaticScratchBytes;
  QuantiserScratch w;
  make_quantiser_scratch(ar, w, n_rows, n_outputs);
  if (ar.failed) {
    lbt::set_error("static scratch too small: %zu bytes, %zu needed", kStaticScratchBytes, ar.used);
    return LBT_ERR_WORKSPACE;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  lbt::ProfScope ps(LBT_PROF_QUANTISE, s, static_cast<double>(n_rows) * n_outputs * (16 + 16 + 8));
  // Nothing of an earlier call's contents is read: every partial sum that is read was written
  // by this call, and find_scales resets the statistics words. The root sums are cleared by a
  // kernel (a memset node would not replay in a captured graph).
  lbt::zero_kernel<<<1, lbt::kThreads, 0, s>>>(reinterpret_cast<uint4*>(root_sums), n_outputs);
  return lbt::run_quantiser(s, g, h, n_rows, n_outputs, row_offset, seed, w.part_a, w.part_b, scales, w.qstats,
                            reinterpret_cast<int2*>(quantised), reinterpret_cast<lbt::I64Pair*>(root_sums));
}

}  // extern "C"

// ---------------------------------------------------------------------------
// The level's stages on the reference's own layouts: the histogram as
// [node - first node of the buffer][output][bin] of (int64 grad, int64 hess)
// (build_tree.h:231-306), the row positions as (node, row) pairs sorted by node
// with the retired rows (node -1) in front (build_tree.cu:997-1001, :1026-1080).
// They run the kernels of lbt_build_tree; what is converted on the way in and
// out is the order (pairs <-> row numbers plus segment starts).
// ---------------------------------------------------------------------------
namespace lbt {
namespace {

// rows[i] = row of pair i
__global__ void __launch_bounds__(kThreads) pairs_to_rows_kernel(const int2* __restrict__ pairs, int64_t n, int32_t* rows)
{
  const int64_t i = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  if (i < n) rows[i] = pairs[i].y;
}

// seg[j] = first pair whose node is >= level_first + j, j = 0 .. n_nodes (the pairs ascend by node)
__global__ void __launch_bounds__(kThreads)
  segment_starts_kernel(const int2* __restrict__ pairs, int64_t n, int level_first, int n_nodes, int32_t* seg)
{
  const int64_t j = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  if (j > n_nodes) return;
  const int64_t want = static_cast<int64_t>(level_first) + j;
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = lo + ((hi - lo) >> 1);
    if (pairs[mid].x < want)
      lo = mid + 1;
    else
      hi = mid;
  }
  seg[j] = static_cast<int32_t>(lo);
}

// block_seg[b] = segment that holds index b * kPartBlock (-1: a retired row); of several segments
// that start at the same index the last one
__global__ void __launch_bounds__(kThreads)
  slab_segments_kernel(const int32_t* __restrict__ seg, int n_nodes, int64_t n_slabs, int32_t* block_seg)
{
  const int64_t b = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  if (b >= n_slabs) return;
  const int64_t i = b * kPartBlock;
  int lo = 0, hi = n_nodes;  // number of starts seg[0 .. n_nodes) that are <= i
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (seg[mid] <= i)
      lo = mid + 1;
    else
      hi = mid;
  }
  block_seg[b] = lo - 1;
}

// every pair that is not of the level (or retired): flag[0] = 1
__global__ void __launch_bounds__(kThreads)
  check_level_kernel(const int2* __restrict__ pairs, int64_t n, int level_first, int level_end, int64_t n_rows,
                     int32_t* flag)
{
  const int64_t i = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  if (i >= n) return;
  const int2 p  = pairs[i];
  const bool ok = (p.x == -1 || (p.x >= level_first && p.x < level_end)) && p.y >= 0 && p.y < n_rows &&
                  (i == 0 || pairs[i - 1].x <= p.x);
  if (!ok) *flag = 1;
}

__global__ void __launch_bounds__(kThreads) bin_feature_kernel(const int32_t* row_pointers, int32_t* bin_feature)
{
  const int f = blockIdx.x;
  for (int b = row_pointers[f] + threadIdx.x; b < row_pointers[f + 1]; b += kThreads) bin_feature[b] = f;
}

template <typename T>
__global__ void __launch_bounds__(kThreads) widen_kernel(const T* in, int64_t n, double* out)
{
  const int64_t i = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  if (i < n) out[i] = static_cast<double>(in[i]);
}

// qstats[0] = max |q| over all 2 * n quantised values (qstats cleared by the caller)
__global__ void __launch_bounds__(kThreads) max_abs_kernel(const int32_t* q, int64_t n2, unsigned long long* qstats)
{
  unsigned long long mx = 0;
  const int64_t stride  = static_cast<int64_t>(gridDim.x) * kThreads;
  for (int64_t i = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x; i < n2; i += stride) {
    const int64_t v              = q[i];
    const unsigned long long a   = static_cast<unsigned long long>(v < 0 ? -v : v);
    mx                           = a > mx ? a : mx;
  }
  for (int off = 32; off >= 1; off >>= 1) {
    const unsigned long long o = __shfl_down(mx, off, 64);
    mx                         = o > mx ? o : mx;
  }
  if ((threadIdx.x & 63) == 0 && mx != 0) atomicMax(&qstats[0], mx);
}

struct HistStageLayout {
  // independent of the level, so that the bin cache of one call is where the next call looks for it
  int32_t* groups;
  int32_t* sgroups;
  int2* bin_lanes;
  RecInfo* rec;
  void* upload_block;
  size_t upload_bytes;
  void* binned;
  size_t binned_bytes;
  uint2* tables;
  void* map_x;
  float* map_t;
  int32_t* straight;
  int32_t* bin_feature;
  unsigned long long* qstats;
  int32_t* flag;
  int32_t* rows;
  int4* tiles;
  LevelMeta* meta;
  LevelMeta* level_total;
  int32_t* pair_sync;
  unsigned long long* partials;
  int32_t* partial_lists;
  int32_t* partial_list_count;
  int32_t* partial_count;
  // sized by the level
  int32_t* seg;
  int32_t* tile_start;
};

void make_hist_stage_layout(Arena& ar, HistStageLayout& L, int64_t N, int F, int S, size_t elem, int level)
{
  const int64_t level_nodes = int64_t(1) << level;
  const size_t upload_at    = ar.used;
  L.groups       = ar.take<int32_t>(F + 1);
  L.sgroups      = ar.take<int32_t>(F + 1);
  L.bin_lanes    = ar.take<int2>(bin_lanes_max(F));
  L.rec          = ar.take<RecInfo>(F);
  L.upload_block = L.groups;
  L.upload_bytes = ar.used - upload_at;
  L.binned_bytes = bin_cache_bytes(N, F, S);
  L.binned       = ar.take<char>(L.binned_bytes + 16);
  L.tables       = ar.take<uint2>(2 * static_cast<size_t>(F) * kMaxCells / 32);
  L.map_x        = ar.take<double>(4 * static_cast<size_t>(F));
  L.map_t        = ar.take<float>(2 * static_cast<size_t>(F));
  L.straight     = ar.take<int32_t>(F);
  L.bin_feature  = ar.take<int32_t>(static_cast<size_t>(F) * S);
  L.qstats       = ar.take<unsigned long long>(2);
  L.flag         = ar.take<int32_t>(4);
  L.rows         = ar.take<int32_t>(N);
  L.tiles        = ar.take<int4>(N / 8 + level_nodes + 1);
  L.meta         = ar.take<LevelMeta>(1);
  L.level_total  = ar.take<LevelMeta>(1);
  L.pair_sync    = ar.take<int32_t>(kPairSyncSlots);
  L.partials     = ar.take<unsigned long long>(static_cast<size_t>(kPartialSlots) * kPartialStrideMax);
  L.partial_lists      = ar.take<int32_t>(static_cast<size_t>(kPartialMaxLists) * kPartialListCap);
  L.partial_list_count = ar.take<int32_t>(kPartialMaxLists);
  L.partial_count      = ar.take<int32_t>(1);
  L.seg        = ar.take<int32_t>(level_nodes + 1);
  L.tile_start = ar.take<int32_t>(level_nodes + 1);
}

struct SplitStageLayout {
  int32_t* bin_feature;  // [bins]
  double* proposals_d;   // [bins]
  int32_t* split_bin;    // [batch_end]
  Cand* partial;         // [nodes of the batch][max(chunks, features)]
};

void make_split_stage_layout(Arena& ar, SplitStageLayout& L, int F, int B, int batch_begin, int batch_end)
{
  const int64_t n_chunks = std::max<int64_t>((static_cast<int64_t>(B) + kSplitChunk - 1) / kSplitChunk, F);
  L.bin_feature = ar.take<int32_t>(B);
  L.proposals_d = ar.take<double>(B);
  L.split_bin   = ar.take<int32_t>(batch_end);
  L.partial     = ar.take<Cand>(static_cast<int64_t>(batch_end - batch_begin) * n_chunks);
}

struct PositionStageLayout {
  int32_t* rows[2];
  int32_t* seg[2];
  int32_t* block_seg[2];
  uint8_t* code;
  int2* block_counts;
  int2* block_offsets;
  int2* seg_prefix;
  int32_t* flag;
};

void make_position_stage_layout(Arena& ar, PositionStageLayout& L, int64_t N, int level)
{
  const int64_t parents = int64_t(1) << level;
  const int64_t slabs   = (N + kPartBlock - 1) / kPartBlock;
  for (int i = 0; i < 2; i++) {
    L.rows[i]      = ar.take<int32_t>(N);
    L.seg[i]       = ar.take<int32_t>(2 * parents + 1);
    L.block_seg[i] = ar.take<int32_t>(slabs);
  }
  L.code          = ar.take<uint8_t>(N);
  L.block_counts  = ar.take<int2>(slabs);
  L.block_offsets = ar.take<int2>(slabs);
  L.seg_prefix    = ar.take<int2>(parents);
  L.flag          = ar.take<int32_t>(4);
}

int stage_batch_ok(int32_t level, int32_t batch_begin, int32_t batch_end)
{
  LBT_REQUIRE(level >= 0 && level <= 24, "level %d out of range [0,24]", level);
  LBT_REQUIRE(batch_begin >= level_begin(level) && batch_end <= level_end(level) && batch_begin < batch_end,
              "nodes [%d, %d) are not a batch of level %d", batch_begin, batch_end, level);
  return LBT_OK;
}

int level_of_node(int node)
{
  int l = 0;
  while (level_end(l) <= node) l++;
  return l;
}

}  // namespace
}  // namespace lbt

extern "C" {

size_t lbt_histogram_level_workspace_bytes(int64_t n_rows, int32_t n_features, int32_t split_samples, int32_t x_dtype,
                                           int32_t level)
{
  if (n_rows < 1 || n_rows >= 2147483647LL || n_features < 1 || level < 0 || level > 24) return 0;
  if (split_samples < 1 || split_samples > LBT_MAX_SPLIT_SAMPLES) return 0;
  if (x_dtype != LBT_F32 && x_dtype != LBT_F64) return 0;
  lbt::Arena ar;
  ar.measure = true;
  lbt::HistStageLayout L{};
  lbt::make_hist_stage_layout(ar, L, n_rows, n_features, split_samples, x_dtype == LBT_F64 ? 8 : 4, level);
  return ar.used + 256;
}

int lbt_histogram_level(void* stream, const void* X, int32_t x_dtype, int64_t n_rows, int32_t n_features,
                        const int32_t* quantised, int32_t n_outputs, const void* proposals,
                        const int32_t* row_pointers, int32_t split_samples, const int32_t* positions, int32_t level,
                        int32_t batch_begin, int32_t batch_end, const int64_t* node_sums, int32_t hist_node_begin,
                        int32_t hist_node_end, int64_t* histogram, void* workspace, size_t workspace_bytes,
                        int32_t reuse_bins)
{
  using namespace lbt;
  LBT_REQUIRE(x_dtype == LBT_F32 || x_dtype == LBT_F64, "unsupported X dtype %d", x_dtype);
  LBT_REQUIRE(n_rows >= 1 && n_rows < 2147483647LL && n_features >= 1 && n_outputs >= 1 && n_outputs <= 65535,
              "bad shape");
  LBT_REQUIRE(split_samples >= 1 && split_samples <= LBT_MAX_SPLIT_SAMPLES, "split_samples must be in [1, %d]",
              LBT_MAX_SPLIT_SAMPLES);
  LBT_REQUIRE(X && quantised && proposals && row_pointers && positions && node_sums && histogram,
              "null input or output pointer");
  LBT_TRY(stage_batch_ok(level, batch_begin, batch_end));
  LBT_REQUIRE(hist_node_begin <= batch_begin && batch_end <= hist_node_end,
              "the histogram buffer [%d, %d) does not hold the batch [%d, %d)", hist_node_begin, hist_node_end,
              batch_begin, batch_end);
  Arena ar;
  LBT_TRY(arena_over(ar, workspace, workspace_bytes));
  HistStageLayout L{};
  const size_t elem = x_dtype == LBT_F64 ? 8 : 4;
  make_hist_stage_layout(ar, L, n_rows, n_features, split_samples, elem, level);
  if (ar.failed) {
    set_error("workspace too small: %zu bytes given, %zu needed", workspace_bytes, ar.used + 256);
    return LBT_ERR_WORKSPACE;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto blocks   = [](int64_t n, int t) { return static_cast<unsigned>((n + t - 1) / t); };
  const int F = n_features, K = n_outputs;
  const int64_t N = n_rows;
  // the bin counts decide the kernels' layout: the one host wait of this call
  std::vector<int32_t> rp(F + 1);
  LBT_HIP(hipMemcpyAsync(rp.data(), row_pointers, sizeof(int32_t) * (F + 1), hipMemcpyDeviceToHost, s));
  LBT_HIP(hipStreamSynchronize(s));
  LBT_REQUIRE(rp[0] == 0, "row_pointers[0] must be 0");
  for (int f = 0; f < F; f++)
    LBT_REQUIRE(rp[f + 1] > rp[f] && rp[f + 1] - rp[f] <= split_samples,
                "feature %d has %d proposals (1 to split_samples = %d expected)", f, rp[f + 1] - rp[f], split_samples);
  const int B = rp[F];

  const int level_first = static_cast<int>(level_begin(level));
  const int level_nodes = 1 << level;
  const int2* pairs     = reinterpret_cast<const int2*>(positions);
  {
    ProfScope ps(LBT_PROF_OTHER, s);
    zero_kernel<<<1, kThreads, 0, s>>>(reinterpret_cast<uint4*>(L.qstats), 1);
    zero_kernel<<<1, kThreads, 0, s>>>(reinterpret_cast<uint4*>(L.flag), 1);
    zero_kernel<<<1, kThreads, 0, s>>>(reinterpret_cast<uint4*>(L.level_total), 2);
    check_level_kernel<<<blocks(N, kThreads), kThreads, 0, s>>>(pairs, N, level_first, level_first + level_nodes, N, L.flag);
    pairs_to_rows_kernel<<<blocks(N, kThreads), kThreads, 0, s>>>(pairs, N, L.rows);
    segment_starts_kernel<<<blocks(level_nodes + 1, kThreads), kThreads, 0, s>>>(pairs, N, level_first, level_nodes, L.seg);
    max_abs_kernel<<<std::min<unsigned>(blocks(N * K * 2, kThreads), 2048u), kThreads, 0, s>>>(quantised, N * K * 2,
                                                                                              L.qstats);
    if (!reuse_bins) bin_feature_kernel<<<F, kThreads, 0, s>>>(row_pointers, L.bin_feature);
  }
  int32_t bad = 0;
  LBT_HIP(hipMemcpyAsync(&bad, L.flag, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  LBT_HIP(hipStreamSynchronize(s));
  LBT_REQUIRE(bad == 0, "positions must be (node, row) pairs sorted by node whose nodes are -1 or of level %d", level);

  HistSetup hs;
  hs.groups = L.groups; hs.sgroups = L.sgroups; hs.tables = L.tables; hs.map_x = L.map_x; hs.map_t = L.map_t; hs.straight = L.straight;
  hs.tile_start = L.tile_start; hs.tiles = L.tiles; hs.binned = L.binned; hs.binned_capacity = L.binned_bytes;
  hs.bin_lanes = L.bin_lanes; hs.rec = L.rec;
  hs.upload_block = L.upload_block; hs.upload_bytes = L.upload_bytes;
  hs.bins_t = nullptr;  // the feature-major copy serves the position updates of a whole build only
  hs.bins_t_stride = 0;
  hs.meta = L.meta; hs.pair_sync = L.pair_sync; hs.partials = L.partials; hs.partial_lists = L.partial_lists;
  hs.partial_list_count = L.partial_list_count; hs.partial_count = L.partial_count; hs.partial_slots = kPartialSlots;
  // the tables are built again on every call (they are small); the cache itself is what reuse_bins keeps
  LBT_TRY(hist_prepare(s, hs, x_dtype == LBT_F64, F, K, N, rp, proposals, row_pointers, X));

  HistBatch hb;
  hb.X = X; hb.F = F; hb.qgh = reinterpret_cast<const int2*>(quantised); hb.K = K; hb.rows = L.rows; hb.seg = L.seg;
  hb.j0 = batch_begin - level_first; hb.n_nodes = batch_end - batch_begin; hb.level_first = level_first;
  hb.proposals = proposals; hb.row_pointers = row_pointers; hb.bin_feature = L.bin_feature;
  hb.hist = HistView{reinterpret_cast<I64Pair*>(histogram), hist_node_begin, hist_node_end, K, B};
  hb.qstats = L.qstats; hb.node_sums = reinterpret_cast<const I64Pair*>(node_sums); hb.level_total = L.level_total;
  hb.n_rows = N; hb.fill_cache = !reuse_bins; hb.identity = false;
  LBT_TRY(hist_launch(s, hs, hb, level));
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

int lbt_scan(void* stream, int64_t* histogram, int32_t hist_node_begin, int32_t hist_node_end, int32_t n_outputs,
             int32_t n_features, const int32_t* row_pointers, int32_t n_bins, const int64_t* node_sums,
             int32_t batch_begin, int32_t batch_end)
{
  using namespace lbt;
  LBT_REQUIRE(histogram && row_pointers && node_sums, "null input or output pointer");
  LBT_REQUIRE(n_features >= 1 && n_outputs >= 1 && n_outputs <= 65535 && n_bins >= n_features, "bad shape");
  LBT_TRY(stage_batch_ok(level_of_node(batch_begin), batch_begin, batch_end));
  LBT_REQUIRE(hist_node_begin <= batch_begin && batch_end <= hist_node_end,
              "the histogram buffer [%d, %d) does not hold the batch [%d, %d)", hist_node_begin, hist_node_end,
              batch_begin, batch_end);
  hipStream_t s = static_cast<hipStream_t>(stream);
  ProfScope ps(LBT_PROF_SCAN, s);
  const HistView hv{reinterpret_cast<I64Pair*>(histogram), hist_node_begin, hist_node_end, n_outputs, n_bins};
  const int n_nodes   = batch_end - batch_begin;
  const int64_t waves = static_cast<int64_t>(n_features) * n_nodes;
  dim3 grid(static_cast<unsigned>((waves + kThreads / 64 - 1) / (kThreads / 64)), n_outputs);
  scan_kernel<<<grid, kThreads, 0, s>>>(hv, reinterpret_cast<const I64Pair*>(node_sums), n_features, row_pointers,
                                        batch_begin, n_nodes, nullptr);
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

size_t lbt_best_split_workspace_bytes(int32_t n_features, int32_t n_bins, int32_t batch_begin, int32_t batch_end)
{
  if (n_features < 1 || n_bins < n_features || batch_begin < 0 || batch_end <= batch_begin) return 0;
  lbt::Arena ar;
  ar.measure = true;
  lbt::SplitStageLayout L{};
  lbt::make_split_stage_layout(ar, L, n_features, n_bins, batch_begin, batch_end);
  return ar.used + 256;
}

int lbt_best_split(void* stream, const int64_t* histogram, int32_t hist_node_begin, int32_t hist_node_end,
                   int32_t n_outputs, int32_t n_features, const void* proposals, int32_t x_dtype,
                   const int32_t* row_pointers, int32_t n_bins, const uint8_t* feature_set, int64_t* node_sums,
                   const double* scales, double l1_regularization, double l2_regularization, double min_split_gain,
                   int32_t batch_begin, int32_t batch_end, double* leaf, int32_t* feature, double* split, double* gain,
                   void* workspace, size_t workspace_bytes)
{
  using namespace lbt;
  LBT_REQUIRE(x_dtype == LBT_F32 || x_dtype == LBT_F64, "unsupported X dtype %d", x_dtype);
  LBT_REQUIRE(histogram && proposals && row_pointers && node_sums && scales && leaf && feature && split && gain,
              "null input or output pointer");
  LBT_REQUIRE(n_features >= 1 && n_outputs >= 1 && n_outputs <= 65535 && n_bins >= n_features, "bad shape");
  LBT_TRY(stage_batch_ok(level_of_node(batch_begin), batch_begin, batch_end));
  LBT_REQUIRE(hist_node_begin <= batch_begin && batch_end <= hist_node_end,
              "the histogram buffer [%d, %d) does not hold the batch [%d, %d)", hist_node_begin, hist_node_end,
              batch_begin, batch_end);
  Arena ar;
  LBT_TRY(arena_over(ar, workspace, workspace_bytes));
  SplitStageLayout L{};
  make_split_stage_layout(ar, L, n_features, n_bins, batch_begin, batch_end);
  if (ar.failed) {
    set_error("workspace too small: %zu bytes given, %zu needed", workspace_bytes, ar.used + 256);
    return LBT_ERR_WORKSPACE;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto blocks   = [](int64_t n, int t) { return static_cast<unsigned>((n + t - 1) / t); };
  ProfScope ps(LBT_PROF_SPLIT, s);
  bin_feature_kernel<<<n_features, kThreads, 0, s>>>(row_pointers, L.bin_feature);
  if (x_dtype == LBT_F64)
    widen_kernel<double><<<blocks(n_bins, kThreads), kThreads, 0, s>>>(static_cast<const double*>(proposals), n_bins,
                                                                      L.proposals_d);
  else
    widen_kernel<float><<<blocks(n_bins, kThreads), kThreads, 0, s>>>(static_cast<const float*>(proposals), n_bins,
                                                                     L.proposals_d);
  // the histogram is only read here; HistView carries it as a mutable pointer for the kernels that fill it
  const HistView hv{reinterpret_cast<I64Pair*>(const_cast<int64_t*>(histogram)), hist_node_begin, hist_node_end,
                    n_outputs, n_bins};
  const int n_nodes  = batch_end - batch_begin;
  const int n_chunks = (n_bins + kSplitChunk - 1) / kSplitChunk;
  dim3 grid(n_nodes, n_chunks);
  split_eval_kernel<<<grid, kThreads, 0, s>>>(hv, reinterpret_cast<const I64Pair*>(node_sums), L.bin_feature,
                                              feature_set, scales, l1_regularization, l2_regularization,
                                              min_split_gain, batch_begin, n_chunks, L.partial);
  split_apply_kernel<<<n_nodes, 64, 0, s>>>(hv, reinterpret_cast<I64Pair*>(node_sums), L.bin_feature, L.proposals_d,
                                            scales, l1_regularization, l2_regularization, batch_begin, n_chunks,
                                            L.partial, leaf, feature, split, gain, row_pointers, L.split_bin, true);
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

size_t lbt_update_positions_workspace_bytes(int64_t n_rows, int32_t level)
{
  if (n_rows < 1 || n_rows >= 2147483647LL || level < 0 || level > 23) return 0;
  lbt::Arena ar;
  ar.measure = true;
  lbt::PositionStageLayout L{};
  lbt::make_position_stage_layout(ar, L, n_rows, level);
  return ar.used + 256;
}

int lbt_update_positions(void* stream, const void* X, int32_t x_dtype, int64_t n_rows, int32_t n_features,
                         int32_t* positions, const int32_t* feature, const double* split, int32_t level,
                         void* workspace, size_t workspace_bytes)
{
  using namespace lbt;
  LBT_REQUIRE(x_dtype == LBT_F32 || x_dtype == LBT_F64, "unsupported X dtype %d", x_dtype);
  LBT_REQUIRE(n_rows >= 1 && n_rows < 2147483647LL && n_features >= 1, "bad shape");
  LBT_REQUIRE(level >= 0 && level <= 23, "level %d out of range [0,23]", level);
  LBT_REQUIRE(X && positions && feature && split, "null input or output pointer");
  Arena ar;
  LBT_TRY(arena_over(ar, workspace, workspace_bytes));
  PositionStageLayout L{};
  make_position_stage_layout(ar, L, n_rows, level);
  if (ar.failed) {
    set_error("workspace too small: %zu bytes given, %zu needed", workspace_bytes, ar.used + 256);
    return LBT_ERR_WORKSPACE;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto blocks   = [](int64_t n, int t) { return static_cast<unsigned>((n + t - 1) / t); };
  const int64_t N       = n_rows;
  const int level_first = static_cast<int>(level_begin(level));
  const int n_parents   = 1 << level;
  const unsigned nb     = blocks(N, kPartBlock);
  int2* pairs           = reinterpret_cast<int2*>(positions);
  {
    ProfScope ps(LBT_PROF_OTHER, s);
    zero_kernel<<<1, kThreads, 0, s>>>(reinterpret_cast<uint4*>(L.flag), 1);
    check_level_kernel<<<blocks(N, kThreads), kThreads, 0, s>>>(pairs, N, level_first, level_first + n_parents, N, L.flag);
    pairs_to_rows_kernel<<<blocks(N, kThreads), kThreads, 0, s>>>(pairs, N, L.rows[0]);
    segment_starts_kernel<<<blocks(n_parents + 1, kThreads), kThreads, 0, s>>>(pairs, N, level_first, n_parents, L.seg[0]);
    slab_segments_kernel<<<blocks(nb, kThreads), kThreads, 0, s>>>(L.seg[0], n_parents, nb, L.block_seg[0]);
  }
  int32_t bad = 0;
  LBT_HIP(hipMemcpyAsync(&bad, L.flag, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  LBT_HIP(hipStreamSynchronize(s));
  LBT_REQUIRE(bad == 0, "positions must be (node, row) pairs sorted by node whose nodes are -1 or of level %d", level);
  ProfScope ps(LBT_PROF_POSITIONS, s);
  if (x_dtype == LBT_F64)
    classify_kernel<double><<<nb, kThreads, 0, s>>>(L.rows[0], N, L.seg[0], L.block_seg[0], n_parents, level_first,
                                                    static_cast<const double*>(X), n_features, feature, split, L.code,
                                                    L.block_counts);
  else
    classify_kernel<float><<<nb, kThreads, 0, s>>>(L.rows[0], N, L.seg[0], L.block_seg[0], n_parents, level_first,
                                                   static_cast<const float*>(X), n_features, feature, split, L.code,
                                                   L.block_counts);
  child_segments_kernel<<<blocks(n_parents, kScanThreads / 64), kScanThreads, 0, s>>>(
    L.seg[0], n_parents, N, L.code, L.block_counts, static_cast<int>(nb), L.block_offsets, L.seg_prefix, L.seg[1],
    L.block_seg[1]);
  scatter_kernel<<<nb, kThreads, 0, s>>>(ScatterArgs{L.rows[0], N, L.code, L.block_offsets, L.seg[0], L.block_seg[0], L.seg_prefix, L.seg[1],
                                                     level_first, n_parents, L.rows[1], nullptr});
  expand_positions_kernel<<<nb, kThreads, 0, s>>>(L.rows[1], N, L.seg[1], L.block_seg[1], 2 * n_parents,
                                                  static_cast<int>(level_begin(level + 1)), pairs);
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

int lbt_build_tree(void* stream, const void* X, int32_t x_dtype, int64_t row_offset,
                   int64_t n_rows, int32_t n_features, const double* g, const double* h,
                   int32_t n_outputs, const uint8_t* feature_set, const lbt_build_params* params,
                   double* leaf, int32_t* feature, double* split, double* gain, double* hessian,
                   void* workspace, size_t workspace_bytes, lbt_build_taps* taps)
{
  return build_tree_entry(stream, X, x_dtype, row_offset, n_rows, n_features, g, h, n_outputs, feature_set, params, leaf,
                          feature, split, gain, hessian, workspace, workspace_bytes, taps, true);
}

int lbt_build_tree_async(void* stream, const void* X, int32_t x_dtype, int64_t row_offset,
                         int64_t n_rows, int32_t n_features, const double* g, const double* h,
                         int32_t n_outputs, const uint8_t* feature_set, const lbt_build_params* params,
                         double* leaf, int32_t* feature, double* split, double* gain, double* hessian,
                         void* workspace, size_t workspace_bytes, lbt_build_taps* taps)
{
  return build_tree_entry(stream, X, x_dtype, row_offset, n_rows, n_features, g, h, n_outputs, feature_set, params, leaf,
                          feature, split, gain, hessian, workspace, workspace_bytes, taps, false);
}

}  // extern "C"
