// BuildTreeTask for inputs of medium size: 2 + 3 * max_depth launches, rows in their own order.
//
// With some ten thousand to a million values per level the builder of lbt_build_tree.hip is a chain of
// ten short launches per level (100,000 x 32: 65 us a level, of which the histogram's atomics are one).
// Here rows stay where they are: a row carries the number of its node, and a level is three launches.
//
//   mid_prologue_kernel   split proposals, one workgroup per feature (build_tree.cu:867-964); chunk sums of
//                         |g| and |h|; the rest clears outputs and state
//   mid_bin_kernel        quantiser and root sums (build_tree.cu:51-204); bins of all values, stored
//                         feature by feature
//   mid_histogram_kernel  a workgroup = (range of rows) x (some features) x (some built nodes) x (output)
//                         with a packed histogram of all those nodes in the LDS, written out whole
//   mid_scan_kernel       a workgroup = (pair of siblings, feature): adds the row ranges' images, running
//                         sums, the sibling as parent minus node, gains (build_tree.cu:597-740); in
//                         wide levels a wave does (mid_scan_waves_kernel)
//   mid_apply_kernel      best features, the nodes' outputs and children (build_tree.cu:740-782), new node
//                         of every row; where few workgroups share a range of rows, the next level's histogram
//                         workgroups do that for themselves instead (a launch less)
//
// The reference leaves a bin as it was accumulated where neither half of its running sum is positive
// (build_tree.cu:645). With hessians that are rounded to 0 or more, that is a bin in front of which no row of
// the node has one, and a sum of grads that is not positive: no split of the node itself, but its sibling
// is the parent minus that bin. The scan keeps to the rule; the histograms are then the reference's as long as it
// keeps the same ones, which it does where those of all levels fit its buffer (zeros_kept). Data with a
// negative rounded hessian, or with one of 0 where they do not fit, take the other builder (see small_tree_build).
// Otherwise a scanned histogram is the running sums everywhere, and it does not matter which ones are kept.
#include <algorithm>
#include <limits>
#include <type_traits>

#include "lbt_device.h"
#include "lbt_internal.h"

namespace lbt {
namespace {

constexpr int kWide     = 1024;  // threads of all kernels but the scan
constexpr int kScan     = 256;
constexpr int kNone     = 0xffff;
constexpr int kRowsBin  = 256;   // rows of a binning tile
template <typename T>
constexpr int kMaxFb    = 128 / sizeof(T);  // features of a binning workgroup: a cache line of a row
constexpr int kRowsApply = 4 * kWide;
constexpr size_t kHistLds = 128 * 1024;
constexpr int64_t kNodesMost = 2500000;  // rows times workgroups that find the nodes of the same ones (nodes_with_histograms)
constexpr int64_t kWavePairs = 1024;     // pairs of siblings times features scanned by a wave each (mid_scan_waves_kernel)
constexpr int kCandsMost     = 4096;     // candidates a histogram workgroup goes through for that (64 KB)

struct MidArgs {
  int N, F, K, S;
  int64_t row_offset;
  int32_t seed;
  int64_t dataset_rows;
  const double* g;
  const double* h;
  const double* chunk_a;  // chunk sums of |g| and |h|, m each
  const double* chunk_b;
  int m;
  const uint8_t* feature_set;
  double l1, l2, min_split_gain;
  int64_t max_nodes;
  int max_depth;
  bool zeros_kept;  // a rounded hessian of 0 (beside a grad) is no reason to take the other builder
  double* leaf;
  int32_t* feature;
  double* split;
  double* gain;
  double* hessian;
  int32_t* row_leaf;
  unsigned long long* answer;  // pinned host memory: flags, and the number of bins, each with `tag` above
  uint32_t tag;
};

// Fixed-order sum of one chunk of up to 4096 entries by 256 threads (see sum_chunk in lbt_build_tree.hip): every thread
// of the workgroup calls it, thread t of each quarter with its own chunk. s_a, s_b: [kWide].
template <bool kAbs>
__device__ __forceinline__ void quarter_sums(const double* __restrict__ a, const double* __restrict__ b, int64_t first,
                                             int64_t n, double* s_a, double* s_b, double* sum_a, double* sum_b)
{
  const int quarter = threadIdx.x >> 8, t = threadIdx.x & 255;
  double xa = 0.0, xb = 0.0;
#pragma unroll 4
  for (int j = 0; j < 16; j++) {
    const int64_t e = first + t + 256 * j;
    if (e < n) {
      xa += kAbs ? fabs(a[e]) : a[e];
      xb += kAbs ? fabs(b[e]) : b[e];
    }
  }
  s_a[quarter * 256 + t] = xa;
  s_b[quarter * 256 + t] = xb;
  __syncthreads();
  for (int stride = 128; stride >= 1; stride >>= 1) {
    if (t < stride) {
      s_a[quarter * 256 + t] += s_a[quarter * 256 + t + stride];
      s_b[quarter * 256 + t] += s_b[quarter * 256 + t + stride];
    }
    __syncthreads();
  }
  *sum_a = s_a[quarter * 256];
  *sum_b = s_b[quarter * 256];
}

template <typename T>
__global__ void __launch_bounds__(kWide)
  mid_prologue_kernel(const T* __restrict__ X, MidArgs a, MidTreeState st, int P, int sum_groups)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ int s_wave[kWide / 64];
  const int block = blockIdx.x, tid = threadIdx.x;
  if (block < a.F) {
    const SampleSpec sp{a.S, a.seed, a.dataset_rows, a.row_offset, a.N, a.F};
    const T* s_prop = nullptr;
    const int n     = feature_proposals<T, kWide>(X, sp, block, P, smem_raw, s_wave, &s_prop);
    const int64_t at = static_cast<int64_t>(block) * a.S;
    for (int i = tid; i < n; i += kWide) {
      // the last proposal becomes +inf (build_tree.cu:953-956)
      const T v = i == n - 1 ? std::numeric_limits<T>::infinity() : s_prop[i];
      static_cast<T*>(st.props)[at + i] = v;
      st.proposals[at + i]              = static_cast<double>(v);
    }
    if (tid == 0) st.counts[block] = n;
    // the cell function and table of the bin search (see build_cells_kernel), a candidate per wave
    __shared__ int s_crowded[kCellMaps];
    __shared__ CellMap<T> s_map[kCellMaps];
    static_assert(kCellMaps <= kWide / 64, "one wave per candidate");
    T* const p = const_cast<T*>(s_prop);
    if (tid == 0) p[n - 1] = std::numeric_limits<T>::infinity();
    __syncthreads();
    if ((tid >> 6) < kCellMaps) {
      const int crowded = crowded_proposals(tid >> 6, p, n, st.cells, tid & 63, &s_map[tid >> 6]);
      if ((tid & 63) == 0) s_crowded[tid >> 6] = crowded;
    }
    __syncthreads();
    int best = 0;
    for (int c = 1; c < kCellMaps; c++)
      if (s_crowded[c] < s_crowded[best]) best = c;
    const CellMap<T> m = s_map[best];
    const float cmax   = static_cast<float>(st.cells - 1);
    const int entries  = st.cells / kCellsPerEntry;
    __shared__ CellScratch s_cells;
    write_cell_entries(p, n, entries, s_cells, st.tables + static_cast<int64_t>(block) * entries,
                       [&](T x) { return cell_of(x, m.scale, m.shift, m.invw, m.nlo, cmax); });
    if (tid == 0) {
      static_cast<T*>(st.map_x)[2 * block]     = m.scale;
      static_cast<T*>(st.map_x)[2 * block + 1] = m.shift;
      st.map_t[2 * block]                      = m.invw;
      st.map_t[2 * block + 1]                  = m.nlo;
    }
    return;
  }
  if (block < a.F + sum_groups) {
    double* s_a = reinterpret_cast<double*>(smem_raw);
    const int c = (block - a.F) * 4 + (tid >> 8);
    double xa, xb;
    quarter_sums<true>(a.g, a.h, static_cast<int64_t>(c) * 4096, static_cast<int64_t>(a.N) * a.K, s_a, s_a + kWide, &xa, &xb);
    if ((tid & 255) == 0 && c < a.m) {
      st.chunk_sums[c]       = xa;
      st.chunk_sums[a.m + c] = xb;
    }
    return;
  }
  const int at         = block - a.F - sum_groups;
  const int64_t stride = static_cast<int64_t>(gridDim.x - a.F - sum_groups) * kWide;
  const int64_t first  = static_cast<int64_t>(at) * kWide + tid;
  for (int64_t i = first; i < a.max_nodes * a.K; i += stride) {
    a.leaf[i]       = 0.0;
    a.hessian[i]    = 0.0;
    st.node_sums[i] = I64Pair{0, 0};
  }
  for (int64_t i = first; i < a.max_nodes; i += stride) {
    a.feature[i] = -1;
    a.split[i]   = 0.0;
    a.gain[i]    = 0.0;
  }
  // all rows start in the root; the places behind the last row belong to no node
  for (int64_t i = first; i < st.pitch; i += stride) st.row_node[0][i] = i < a.N ? 0 : kNone;
  if (first <= a.max_depth) st.live[first] = first == 0 ? 1 : 0;
  if (first < 4) st.q_stats[first] = 0;
}

struct BinPlan {
  int quant_groups;  // workgroups of the quantiser
  int quant_per;     // entries that one of them rounds, a multiple of kWide
  int fb;            // features of a binning workgroup
  int fb_log;        // lanes per row, log2
  int n_fb;          // feature blocks
  int row_groups;    // workgroups that share the row tiles of a feature block
  int search_steps;  // of a binary search over a feature's proposals
};

// LDS elements per feature: the proposals, the +inf entries a window of probes may touch, and an odd pitch
__host__ __device__ constexpr int prop_pitch(int S) { return (S + 8) | 1; }

// What bounds it is latency: a few tiles per workgroup behind a chain of launch, tables and first rows, and the quantiser's own
// chain beside it. With the first rows asked for before the tables, all of a thread's loads of these under way together, the searches side by
// side and 1024 entries to a workgroup of the quantiser 100,000 x 32 takes 11 us (20.5), 250,000 x 43 30 (41), 1,500,000 x 33 118 (150),
// 1,304,790 x 26 in double with 3 outputs 116 (166). Two workgroups to a CU: 64 registers.
template <typename T, typename BinT>
__global__ void __launch_bounds__(kWide, 8)
  mid_bin_kernel(const T* __restrict__ X, MidArgs a, MidTreeState st, BinPlan p)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int tid = threadIdx.x;
  if (static_cast<int>(blockIdx.x) < p.quant_groups) {
    // the scales, formed by every workgroup in the same fixed order, then this workgroup's entries
    double* s_a = reinterpret_cast<double*>(smem_raw);
    __shared__ unsigned long long s_sum[2 * kMidMaxOutputs + 2];
    __shared__ unsigned s_flags;
    if (tid < 2 * a.K + 2) s_sum[tid] = 0;
    if (tid == 0) s_flags = 0;
    double sum_a, sum_b;
    if (a.m > 1) {
      quarter_sums<false>(a.chunk_a, a.chunk_b, 0, a.m, s_a, s_a + kWide, &sum_a, &sum_b);
    } else {
      __syncthreads();
      sum_a = a.chunk_a[0];
      sum_b = a.chunk_b[0];
    }
    const double max_int = 2147483647.0;
    const double sg = sum_a == 0 ? 1 : max_int / sum_a, sh = sum_b == 0 ? 1 : max_int / sum_b;
    if (blockIdx.x == 0 && tid == 0) {
      st.scales[0] = sg;
      st.scales[1] = sh;
      st.scales[2] = 1.0 / sg;
      st.scales[3] = 1.0 / sh;
    }
    if (blockIdx.x == 0) {
      // first bin of every feature among all bins
      __shared__ int s_wave[kWide / 64];
      const int per = (a.F + kWide - 1) / kWide, f0 = min(a.F, tid * per), f1 = min(a.F, f0 + per);
      int mine = 0;
      for (int f = f0; f < f1; f++) mine += st.counts[f];
      int run = block_exclusive_sum32<kWide>(mine, s_wave);
      for (int f = f0; f < f1; f++) {
        st.rp[f] = run;
        run += st.counts[f];
      }
      if (tid == kWide - 1) st.rp[a.F] = run;
    }
    const int64_t n  = static_cast<int64_t>(a.N) * a.K;
    const int64_t e0 = static_cast<int64_t>(blockIdx.x) * p.quant_per, e1 = e0 + p.quant_per < n ? e0 + p.quant_per : n;
    int64_t sum_g = 0, sum_h = 0;
    unsigned long long up = 0, down = 0;
    unsigned flags = 0;
    double grad = 0.0, hess = 0.0;
    if (e0 + tid < e1) {
      grad = a.g[e0 + tid];
      hess = a.h[e0 + tid];
    }
    for (int64_t e = e0 + tid; e < e1; e += kWide) {
      const double g = grad, h = hess;
      if (e + kWide < e1) {
        grad = a.g[e + kWide];
        hess = a.h[e + kWide];
      }
      const int64_t row = a.K == 1 ? e : e / a.K;
      const int k       = a.K == 1 ? 0 : static_cast<int>(e - row * a.K);
      int64_t qg, qh;
      quantise_pair(g, h, sg, sh, static_cast<int64_t>(a.seed), row + a.row_offset, k, &qg, &qh);
      if (qg > 2147483647LL || qg < -2147483647LL || qh > 2147483647LL || qh < -2147483647LL) flags |= 2u;
      if (qh < 0 || (qh == 0 && qg != 0 && !a.zeros_kept)) flags |= 1u;
      st.q[static_cast<int64_t>(k) * st.pitch + row] = make_int2(static_cast<int>(qg), static_cast<int>(qh));
      up += qg > 0 ? static_cast<unsigned long long>(qg) : 0ULL;
      down += qg < 0 ? static_cast<unsigned long long>(-qg) : 0ULL;
      if (a.K == 1) {
        sum_g += qg;
        sum_h += qh;
      } else {
        atomicAdd(&s_sum[2 * k], static_cast<unsigned long long>(qg));
        atomicAdd(&s_sum[2 * k + 1], static_cast<unsigned long long>(qh));
      }
    }
    const int64_t wu = wave_inclusive_sum(static_cast<int64_t>(up)), wd = wave_inclusive_sum(static_cast<int64_t>(down));
    sum_g = wave_inclusive_sum(sum_g);
    sum_h = wave_inclusive_sum(sum_h);
    if ((tid & 63) == 63) {
      if (a.K == 1) {
        atomicAdd(&s_sum[0], static_cast<unsigned long long>(sum_g));
        atomicAdd(&s_sum[1], static_cast<unsigned long long>(sum_h));
      }
      atomicAdd(&s_sum[2 * a.K], static_cast<unsigned long long>(wu));
      atomicAdd(&s_sum[2 * a.K + 1], static_cast<unsigned long long>(wd));
    }
    if (flags != 0) atomicOr(&s_flags, flags);
    __syncthreads();
    if (tid < a.K) {
      atomic_add_i64(&st.node_sums[tid].grad, static_cast<int64_t>(s_sum[2 * tid]));
      atomic_add_i64(&st.node_sums[tid].hess, static_cast<int64_t>(s_sum[2 * tid + 1]));
    }
    if (tid == 0) {
      atomicAdd(&st.q_stats[0], s_sum[2 * a.K]);
      atomicAdd(&st.q_stats[1], s_sum[2 * a.K + 1]);
      if (s_flags != 0) atomicOr(&st.q_stats[2], static_cast<unsigned long long>(s_flags));
    }
    return;
  }
  // binning: proposals and tables of the block's features in the LDS (odd pitches: the lanes of a row start in
  // different banks), a tile of rows at a time, turned in the LDS and stored feature by feature
  const int block = static_cast<int>(blockIdx.x) - p.quant_groups;
  const int fblk = block % p.n_fb, rg = block / p.n_fb;
  const int f0 = fblk * p.fb, nf = min(p.fb, a.F - f0);
  const int pitch = prop_pitch(a.S), entries = st.cells / kCellsPerEntry, tpitch = entries | 1;
  uint2* s_table = reinterpret_cast<uint2*>(smem_raw);            // [fb][tpitch]
  T* s_prop      = reinterpret_cast<T*>(s_table + p.fb * tpitch);  // [fb][pitch]
  int* s_n       = reinterpret_cast<int*>(s_prop + static_cast<size_t>(p.fb) * pitch);
  constexpr int kTilePitch = kRowsBin + 4 / sizeof(BinT);
  BinT* s_bin       = reinterpret_cast<BinT*>(s_n + p.fb);  // [fb][kTilePitch]
  const int fi = tid & ((1 << p.fb_log) - 1), r_first = tid >> p.fb_log, r_step = kWide >> p.fb_log;
  const int fm = f0 + min(fi, nf - 1);  // lanes without a feature of their own search the last one's values
  const int tiles = (a.N + kRowsBin - 1) / kRowsBin;
  // A thread's values of a tile: on their way while the tables come into the LDS, or while the tile before is written.
  constexpr int kMost  = kRowsBin * kMaxFb<T> / kWide;
  constexpr int kBatch = sizeof(T) == 4 ? 4 : 2;  // values searched side by side
  T x[kMost];
  // (Few features: fewer turns, and of one or two features waves that have no rows. Taken all the same they were 1.2 to 1.6 times the pass, f32:
  // 4,000,000 x 1 63 us, x 2 73, x 4 100; 112, 114 and 117 with all of them.)
  const bool has_rows = r_first < kRowsBin;
  auto fetch          = [&](int tile) {
    if (!has_rows) return;
#pragma unroll
    for (int u0 = 0; u0 < kMost; u0 += kBatch) {
      if (u0 * r_step >= kRowsBin) break;
#pragma unroll
      for (int u = u0; u < u0 + kBatch; u++) {
        const int r       = min(r_first + u * r_step, kRowsBin - 1);
        const int64_t row = min(static_cast<int64_t>(tile) * kRowsBin + r, static_cast<int64_t>(a.N) - 1);
        x[u]              = X[row * a.F + fm];
      }
    }
  };
  fetch(rg);
  for (int i = tid; i < nf; i += kWide) s_n[i] = st.counts[f0 + i];
  // a feature per half wave, what lies behind its last proposal is set apart below
  {
    const int half = tid >> 5, j0 = tid & 31;
    for (int c = half; c < nf; c += kWide / 32) {
      const uint2* src = st.tables + static_cast<int64_t>(f0 + c) * entries;
      const T* from    = static_cast<const T*>(st.props) + static_cast<int64_t>(f0 + c) * a.S;
      uint2 e[2];
      T v[8];
      for (int b = 0; b < max(entries, (a.S + 3) / 4); b += 64) {  // 64 entries and 256 samples under way at once
#pragma unroll
        for (int u = 0; u < 2; u++) e[u] = src[min(b + j0 + 32 * u, entries - 1)];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = from[min(4 * b + j0 + 32 * u, a.S - 1)];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 2; u++)
          if (b + j0 + 32 * u < entries) s_table[c * tpitch + b + j0 + 32 * u] = e[u];
#pragma unroll
        for (int u = 0; u < 8; u++)
          if (4 * b + j0 + 32 * u < a.S) s_prop[c * pitch + 4 * b + j0 + 32 * u] = v[u];
      }
    }
  }
  __syncthreads();
  // +inf from the last proposal on, for the probes that run past it
  for (int i = tid; i < nf * 8; i += kWide) s_prop[(i >> 3) * pitch + s_n[i >> 3] - 1 + (i & 7)] = std::numeric_limits<T>::infinity();
  const T scale = static_cast<const T*>(st.map_x)[2 * fm], shift = static_cast<const T*>(st.map_x)[2 * fm + 1];
  const float invw = st.map_t[2 * fm], nlo = st.map_t[2 * fm + 1], cmax = static_cast<float>(st.cells - 1);
  BinT* const out = static_cast<BinT*>(st.bins);
  const T* prop      = s_prop + min(fi, nf - 1) * pitch;
  const uint2* table = s_table + min(fi, nf - 1) * tpitch;
  for (int tile = rg; tile < tiles; tile += p.row_groups) {
    __syncthreads();
    // the searches of a batch go stage by stage, as in bin_rows_kernel: the table's entries, three probes at once, and for the
    // few lanes that need more four further ones and a binary search
#pragma unroll
    for (int u0 = 0; u0 < kMost; u0 += kBatch) {
      if (!has_rows || u0 * r_step >= kRowsBin) break;
      int bn[kBatch], cell[kBatch];
      uint2 entry[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; u++) {
        cell[u]  = cell_of(x[u0 + u], scale, shift, invw, nlo, cmax);
        entry[u] = table[static_cast<unsigned>(cell[u]) >> kCellShift];
      }
      __builtin_amdgcn_sched_barrier(0);
      T probe[kBatch][3];
#pragma unroll
      for (int u = 0; u < kBatch; u++) {
        bn[u] = table_start(entry[u], cell[u]);
#pragma unroll
        for (int i = 0; i < 3; i++) probe[u][i] = prop[bn[u] + i];
      }
      __builtin_amdgcn_sched_barrier(0);
      bool more = false;
#pragma unroll
      for (int u = 0; u < kBatch; u++) {
        const T v = x[u0 + u];
        bn[u] += (probe[u][0] < v ? 1 : 0) + (probe[u][1] < v ? 1 : 0) + (probe[u][2] < v ? 1 : 0);
        more = more || probe[u][2] < v;
      }
      if (__any(more)) {
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
          const T v   = x[u0 + u];
          const T* pp = prop + bn[u];
          if (!__any(pp[0] < v)) continue;
          const int c2 = (pp[0] < v ? 1 : 0) + (pp[1] < v ? 1 : 0) + (pp[2] < v ? 1 : 0) + (pp[3] < v ? 1 : 0);
          bn[u] += c2;
          if (__any(c2 == 4)) bn[u] += count_less(pp + 4, c2 == 4 ? s_n[min(fi, nf - 1)] - bn[u] : 0, v, p.search_steps);
        }
      }
#pragma unroll
      for (int u = 0; u < kBatch; u++) {
        const int r = r_first + (u0 + u) * r_step;
        if (fi < nf && r < kRowsBin) s_bin[fi * kTilePitch + r] = static_cast<BinT>(bn[u]);
      }
    }
    if (tile + p.row_groups < tiles) fetch(tile + p.row_groups);
    __syncthreads();
    constexpr int kPer = 4 / sizeof(BinT);  // bins per word
    for (int i = tid; i < nf * (kRowsBin / kPer); i += kWide) {
      const int c = i / (kRowsBin / kPer), w = i - c * (kRowsBin / kPer);
      *reinterpret_cast<uint32_t*>(out + static_cast<int64_t>(f0 + c) * st.pitch + static_cast<int64_t>(tile) * kRowsBin + w * kPer) =
        *reinterpret_cast<const uint32_t*>(s_bin + c * kTilePitch + w * kPer);
    }
  }
}

// Nothing to do at a level: no node was split into it, or (known at the root) the data are for the other builder.
__device__ __forceinline__ bool level_is_empty(const MidTreeState& st, int depth)
{
  return st.live[depth] == 0 || (depth == 0 && st.q_stats[2] != 0);
}

// How a level's histograms are dealt to workgroups.
struct LevelPlan {
  int depth, level_first, n_nodes;
  int built;        // nodes whose histogram is accumulated: one of every pair
  int fw, n_fb;     // features per workgroup, blocks of them
  int bw, n_bb;     // built nodes per workgroup, blocks of them
  int chunks;       // row ranges
  int chunk_rows;   // multiple of 4
  bool pairs;       // two workgroups share a CU
  bool last;
};

// Features of a histogram workgroup at most. Eight share a row's node and pair among more bins but fill the feature
// blocks worse and leave half as many of them: with eight from 150,000 rows on, 300,000 x 43, depth 8 took 360 us (340 with
// four), 1,000,000 x 50 with 512 samples 802 (737), 150,000 x 20 with 4 outputs 273 (243), 300,000 x 32 the same.
constexpr int kMaxFw = 4;

// Values (rows times features and outputs) up to which it is the images of the row ranges that cost, not the additions: a scan
// workgroup reads 64 KB of them with 32 ranges, which takes it 6000 of 14,000 cycles however many loads are under way. One
// workgroup for every CU then, not two, and two features each instead of four (with several outputs the ranges are few anyway): fewer
// ranges. Fits with two workgroups and with one, us: 20,000 x 100, depth 6, 5 rounds 1040 and 945; 9000 x 200, depth 5 945 and 825; 250,000 x 43,
// depth 8 1965 and 1890; 300,000 x 16 with 128 samples 1060 and 1005; 60,000 x 20 with 4 outputs 1235 and 1110. Trees of depth 6 with 256
// samples just below the line: 595,000 x 20 227 and 205, 119,000 x 100 228 and 218, 29,750 x 400 283 and 275; with 64, whose images are a
// quarter, 209 and 190, 197 and 197, 47,600 x 250 208 and 211. Above it, not taken: 240,000 x 100 270 and 273, 400,000 x 45 with 64 samples
// 219 and 231, 60,000 x 300 285 and 304, 100,000 x 40 with 4 outputs and 128 samples 227 and 234; few columns would still gain (1,000,000 x
// 20, depth 8 365 and 344).
constexpr int64_t kImageValues = 12000000;

// Which of a pair of siblings is accumulated (build_tree.h:92-104).
__device__ __forceinline__ int built_of_pair(const I64Pair* __restrict__ node_sums, int level_first, int pair, int K)
{
  const int64_t hl = node_sums[static_cast<int64_t>(level_first + 2 * pair) * K].hess;
  const int64_t hr = node_sums[static_cast<int64_t>(level_first + 2 * pair + 1) * K].hess;
  return hl < hr ? 2 * pair : 2 * pair + 1;
}

// Beside the bin of a candidate: its left child has the smaller hessian of the two, and is the one that is accumulated.
constexpr int kLeftSmaller = 1 << 30;

// The split of node j of the level by 1 << lanes_log lanes of a wave (`sub` numbers them), and, if `write`,
// what follows from it: the node's outputs, its children's sums and leaf values. x: feature, -1 for a leaf;
// y: its last bin that goes left (kLeftSmaller with it: see there). Lanes whose j is no node call it too (j < 0).
__device__ __forceinline__ int2 decide_node(const MidArgs& a, const MidTreeState& st, const LevelPlan& p, int j, int sub,
                                            int lanes, bool write)
{
  const int node = p.level_first + j;
  double best    = 0.0;
  unsigned key   = 0;
  int ft = 0, rel = 0;
  auto take = [&](double gain_o, unsigned key_o, int ft_o, int rel_o) {
    const bool better = gain_o > best || (gain_o == best && key_o > key);
    best = better ? gain_o : best;
    key  = better ? key_o : key;
    ft   = better ? ft_o : ft;
    rel  = better ? rel_o : rel;
  };
  const bool here = j >= 0 && st.node_sums[static_cast<int64_t>(node) * a.K].hess > 0;
  if (here) {
    const SmallCand* c = st.cand + static_cast<int64_t>(j) * a.F;
    for (int i = sub; i < a.F; i += lanes) {
      const SmallCand o = c[i];
      take(o.gain, o.key, i, o.rel);
    }
  }
  if (lanes == 64) wave_best_split(best, key, ft, rel);
  for (int off = lanes == 64 ? 0 : lanes >> 1; off >= 1; off >>= 1) {
    const double g   = __shfl_xor(best, off, 64);
    const unsigned o = static_cast<unsigned>(__shfl_xor(static_cast<int>(key), off, 64));
    const int f_o = __shfl_xor(ft, off, 64), r_o = __shfl_xor(rel, off, 64);
    take(g, o, f_o, r_o);
  }
  const bool splits = here && key != 0 && best > 1e-5;
  if (write && j >= 0) {
    const double inv_g = st.scales[2], inv_h = st.scales[3];
    if (p.depth == 0)
      for (int k = sub; k < a.K; k += lanes) {
        const I64Pair ns = st.node_sums[k];
        const double G = static_cast<double>(ns.grad) * inv_g, H = static_cast<double>(ns.hess) * inv_h;
        a.leaf[k]      = calculate_leaf_value(G, H, a.l1, a.l2);
        a.hessian[k]   = H;
      }
    if (splits) {
      const int64_t fs = static_cast<int64_t>(a.F) * a.S;
      const int lc = left_child(node), rc = right_child(node);
      // (the last level of one output stores no histograms)
      const uint2* h = p.last && a.K == 1 ? st.left + static_cast<int64_t>(j) * a.F + ft
                                          : st.hist[p.depth & 1] + static_cast<int64_t>(j) * a.K * fs + static_cast<int64_t>(ft) * a.S + (rel & ~kLeftSmaller);
      const uint32_t down = static_cast<uint32_t>(st.q_stats[1]);
      for (int k = sub; k < a.K; k += lanes) {
        const int64_t at = static_cast<int64_t>(node) * a.K + k, l = static_cast<int64_t>(lc) * a.K + k,
                      r = static_cast<int64_t>(rc) * a.K + k;
        const I64Pair ns = st.node_sums[at];
        const uint2 low  = h[k * fs];
        const I64Pair ls{static_cast<int64_t>(low.x + down) - static_cast<int64_t>(down), static_cast<int64_t>(low.y)};
        const I64Pair rs{ns.grad - ls.grad, ns.hess - ls.hess};
        const double lg = static_cast<double>(ls.grad) * inv_g, lh = static_cast<double>(ls.hess) * inv_h;
        const double rg = static_cast<double>(rs.grad) * inv_g, rh = static_cast<double>(rs.hess) * inv_h;
        st.node_sums[l] = ls;
        st.node_sums[r] = rs;
        a.leaf[l]       = calculate_leaf_value(lg, lh, a.l1, a.l2);
        a.leaf[r]       = calculate_leaf_value(rg, rh, a.l1, a.l2);
        a.hessian[l]    = lh;
        a.hessian[r]    = rh;
      }
      if (sub == 0) {
        a.feature[node] = ft;
        a.split[node]   = st.proposals[static_cast<int64_t>(ft) * a.S + (rel & ~kLeftSmaller)];
        a.gain[node]    = best;
        st.live[p.depth + 1] = 1;
      }
    }
  }
  return make_int2(splits ? ft : -1, rel);
}

// Four rows in a row, from r on, in the nodes node[] of a level (kNone: in none) with the splits s_split: their nodes of the
// next level, kNone where a row ends.
template <typename BinT>
struct RowSplits {
  unsigned next[4];
  int2 sp[4];
  __device__ __forceinline__ RowSplits(const MidArgs& a, const MidTreeState& st, const int2* s_split, const unsigned (&node)[4], int r)
  {
    const BinT* const bins = static_cast<const BinT*>(st.bins);
    int bin[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      sp[u]  = node[u] != kNone ? s_split[node[u]] : make_int2(-1, 0);
      bin[u] = sp[u].x >= 0 ? static_cast<int>(bins[static_cast<int64_t>(sp[u].x) * st.pitch + r + u]) : 0;
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
      next[u] = sp[u].x >= 0 ? 2 * node[u] + (bin[u] <= (sp[u].y & ~kLeftSmaller) ? 0u : 1u) : kNone;
  }
  // the nodes in which rows end: all of them at the last level
  __device__ __forceinline__ void store_leaves(const MidArgs& a, const LevelPlan& p, const unsigned (&node)[4], int r, bool last) const
  {
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (a.row_leaf != nullptr && node[u] != kNone && (sp[u].x < 0 || last))
        a.row_leaf[r + u] = sp[u].x < 0 ? p.level_first + static_cast<int>(node[u]) : 2 * p.level_first + 1 + static_cast<int>(next[u]);
  }
};

// Where a level's histogram workgroups take the rows' nodes from. kCarried: row_node holds this level's. kDecide: it holds the
// parents', whose splits every workgroup finds for itself. kDecided: the same with the splits of mid_decide_kernel.
// Finding splits and bins takes a workgroup two loads one after the other (2 us), a launch of mid_apply_kernel 6 to 7.
enum class Nodes { kCarried, kDecide, kDecided };

// A packed word holds the sum of grads in its upper and the sum of hessians in its lower half. Rounded
// hessians are not negative here and sum up to less than 2^32. The grads of all rows sum up to -down and +up
// with up + down < 2^32, so the lower half of a sum + down is the sum + down (mid_scan_kernel).
template <typename BinT, Nodes kNodes>
__global__ void __launch_bounds__(kWide)
  mid_histogram_kernel(MidArgs a, MidTreeState st, LevelPlan p, LevelPlan above, int lanes_log, int writers,
                       const uint16_t* __restrict__ from, uint16_t* __restrict__ to)
{
  constexpr bool kCarried = kNodes == Nodes::kCarried;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  unsigned long long* s_hist = reinterpret_cast<unsigned long long*>(smem_raw);  // [fw][bw][S]
  __shared__ uint16_t s_slot[kMidMaxLevelNodes];                                 // node -> its histogram here, kNone: none
  __shared__ int2 s_split[kCarried ? 1 : kMidMaxLevelNodes / 2];                 // of the parents
  const int tid = threadIdx.x;
  if (kNodes == Nodes::kDecide && static_cast<int>(blockIdx.x) < writers) {
    // what follows from the parents' splits
    if (level_is_empty(st, above.depth)) return;
    const int j = static_cast<int>(blockIdx.x * kWide + threadIdx.x) >> lanes_log;
    decide_node(a, st, above, j < above.n_nodes ? j : -1, tid & ((1 << lanes_log) - 1), 1 << lanes_log, true);
    return;
  }
  const int block = static_cast<int>(blockIdx.x) - writers;
  // ranges of rows vary fastest over the XCDs, so that one range's workgroups share an L2
  const int lanes8 = p.chunks >= 8 ? 8 : 1;
  const int low = block % lanes8;
  int rest      = block / lanes8;
  const int inner = p.n_fb * p.n_bb * a.K;
  const int chunk = rest / inner * lanes8 + low;
  rest            = rest % inner;
  if (chunk >= p.chunks) return;
  const int k = rest % a.K, fb = rest / a.K % p.n_fb, bb = rest / a.K / p.n_fb;
  const bool empty = level_is_empty(st, kCarried ? p.depth : above.depth);
  if (p.depth == 0 && blockIdx.x == 0 && tid == 0) {
    __hip_atomic_store(a.answer + 1, (static_cast<unsigned long long>(a.tag) << 32) | static_cast<unsigned>(st.rp[a.F]),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(a.answer, (static_cast<unsigned long long>(a.tag) << 32) | st.q_stats[2], __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  }
  if (empty) return;
  const int f0 = fb * p.fw, nf = min(p.fw, a.F - f0);
  const int b0 = bb * p.bw, nb = min(p.bw, p.built - b0);
  if constexpr (kNodes == Nodes::kDecided)
    for (int j = tid; j < above.n_nodes; j += kWide) s_split[j] = st.splits[j];
  if constexpr (kNodes == Nodes::kDecide) {
    const int lanes = 1 << lanes_log, sub = tid & (lanes - 1);
    for (int j0 = 0; j0 < above.n_nodes; j0 += kWide >> lanes_log) {
      const int j   = j0 + (tid >> lanes_log);
      const int2 sp = decide_node(a, st, above, j < above.n_nodes ? j : -1, sub, lanes, false);
      if (sub == 0 && j < above.n_nodes) s_split[j] = sp;
    }
  }
  if constexpr (!kCarried) __syncthreads();
  for (int j = tid; j < p.n_nodes; j += kWide) {
    int slot = kNone;
    if constexpr (!kCarried) {
      const int2 sp = s_split[j / 2];
      if (j / 2 >= b0 && j / 2 < b0 + nb && sp.x >= 0 && (j & 1) == ((sp.y & kLeftSmaller) != 0 ? 0 : 1)) slot = j / 2 - b0;
    } else if (p.depth == 0)
      slot = 0;
    else if (j / 2 >= b0 && j / 2 < b0 + nb && built_of_pair(st.node_sums, p.level_first, j / 2, a.K) == j)
      slot = j / 2 - b0;
    s_slot[j] = static_cast<uint16_t>(slot);
  }
  for (int i = tid; i < p.fw * p.bw * a.S; i += kWide) s_hist[i] = 0;
  __syncthreads();
  const int r_begin = chunk * p.chunk_rows, r_end = min(a.N, r_begin + p.chunk_rows);
  const BinT* const bins = static_cast<const BinT*>(st.bins) + static_cast<int64_t>(f0) * st.pitch;
  const int2* const q    = st.q + static_cast<int64_t>(k) * st.pitch;
  for (int r = r_begin + 4 * tid; r < r_end; r += 4 * kWide) {
    const uint2 nd = *reinterpret_cast<const uint2*>(from + r);
    const uint4 qa = *reinterpret_cast<const uint4*>(q + r), qb = *reinterpret_cast<const uint4*>(q + r + 2);
    uint32_t w[kMaxFw][sizeof(BinT)];
#pragma unroll
    for (int i = 0; i < kMaxFw; i++)
      if (i < nf) {
        const uint32_t* src = reinterpret_cast<const uint32_t*>(bins + static_cast<int64_t>(i) * st.pitch + r);
#pragma unroll
        for (int u = 0; u < static_cast<int>(sizeof(BinT)); u++) w[i][u] = src[u];
      }
    unsigned node[4] = {nd.x & 0xffffu, nd.x >> 16, nd.y & 0xffffu, nd.y >> 16};
    if constexpr (!kCarried) {
      const RowSplits<BinT> rows(a, st, s_split, node, r);
      if (fb == 0 && bb == 0 && k == 0) {
        *reinterpret_cast<uint2*>(to + r) = make_uint2(rows.next[0] | rows.next[1] << 16, rows.next[2] | rows.next[3] << 16);
        rows.store_leaves(a, above, node, r, false);
      }
#pragma unroll
      for (int u = 0; u < 4; u++) node[u] = rows.next[u];
    }
    const uint32_t qg[4] = {qa.x, qa.z, qb.x, qb.z}, qh[4] = {qa.y, qa.w, qb.y, qb.w};
#pragma unroll
    for (int u = 0; u < 4; u++) {
      // (rows past the last one belong to no node; a row past the chunk's end is the next chunk's)
      const int slot = node[u] != kNone && r + u < r_end ? s_slot[node[u]] : kNone;
      if (slot != kNone) {
        const unsigned long long word = (static_cast<unsigned long long>(qg[u]) << 32) | qh[u];
        unsigned long long* h         = s_hist + slot * a.S;
#pragma unroll
        for (int i = 0; i < kMaxFw; i++)
          if (i < nf) {
            const unsigned bin = sizeof(BinT) == 1 ? (w[i][0] >> (8 * u)) & 0xffu
                                                   : (w[i][(u >> 1) & (sizeof(BinT) - 1)] >> (16 * (u & 1))) & 0xffffu;
            atomicAdd(h + static_cast<int64_t>(i) * p.bw * a.S + bin, word);
          }
      }
    }
  }
  __syncthreads();
  // the image of this range of rows: [built node][output][feature][bin]
  unsigned long long* image =
    st.images + ((static_cast<int64_t>(chunk) * p.built + b0) * a.K + k) * static_cast<int64_t>(a.F) * a.S + static_cast<int64_t>(f0) * a.S;
  for (int b = 0; b < nb; b++)
    for (int i = tid; i < nf * a.S; i += kWide) {
      const int fi = i / a.S, bin = i - fi * a.S;
      image[static_cast<int64_t>(b) * a.K * a.F * a.S + i] = s_hist[(fi * p.bw + b) * a.S + bin];
    }
}

// A launch of a narrow level is a chain of latencies: the images, the sums over the workgroup, the quotients, the best
// bin. The quotients of a node and its sibling therefore have no branch between them, the nodes' sums are asked for with
// the images, and the best of a wave is found without the LDS (18 permutes one after the other, twice): the eight levels
// of 250,000 x 43 took 90 us, now 79; the six of 100,000 x 32 50 and 43. All loads in front of the first wait
// instead, with the terms that do not depend on the bin formed once, was slower: 8.3 to 9.5 us a narrow level where it
// had been 7.5 to 8.1.
// kLess: kLeftSmaller beside the candidates' bins, for histogram workgroups that decide (42.2 us a launch on 5000 x 200 with 8 outputs, depth 5, to
// 41.1 without).
// Histograms in memory are the lower halves of their sums, 8 bytes a bin, and the last level of one output (kLast) stores none, only what lies left of a
// feature's best split. (Where the rule on zeros left a bin as it was in the parent, which has no hessian then, what a sibling keeps there can lie
// outside of -down and up; no node below takes a split at it, and what is subtracted from it is exact in 32 bits.) With 16 bytes, and all levels
// stored, the two deepest levels of 50,000 x 200, depth 8, took 33 and 61 us: now 18 and 28, by waves (mid_scan_waves_kernel).
// kAhead: with several outputs a workgroup's sums of the images are asked for one output ahead, all ranges of rows that
// kAhead holds at once. A chain of loads, sums and barriers per output took 2.5 us an output (400,000 x 12 with 8 outputs and 32
// ranges: 20 us a narrow level, now 16; 11,094 x 120 with 5 outputs, 512 samples, depth 8: a tree in 754 us, now 635). As many
// loads as there are ranges, up to 16: 16 always took 5000 x 200 with 8 outputs, which has 4, from 209 to 221 us, 4 take 198.
template <bool kLess, bool kLast, int kAhead>
__global__ void __launch_bounds__(kScan)
  mid_scan_kernel(MidArgs a, MidTreeState st, LevelPlan p)
{
  __shared__ uint2 s_tot[2][kScan / 64];
  __shared__ uint2 s_carry[kMidMaxOutputs];
  __shared__ double s_best[2][kScan / 64];
  __shared__ unsigned s_bkey[2][kScan / 64];
  __shared__ int s_less[2][kScan / 64];
  __shared__ uint2 s_cell[kLast ? 2 : 1][kScan / 64];
  const int f = blockIdx.x % a.F, pair = blockIdx.x / a.F;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  if (level_is_empty(st, p.depth)) return;
  const bool usable = a.feature_set == nullptr || a.feature_set[f] != 0;
  const int left    = 2 * pair;
  const bool root   = p.depth == 0;
  // the children of a node that did not split have no rows
  if (!root && st.node_sums[static_cast<int64_t>(p.level_first + left) * a.K].hess <= 0) return;
  const int node = root ? 0 : built_of_pair(st.node_sums, p.level_first, pair, a.K);
  const int sib  = root ? 0 : node ^ 1;
  if (!usable) {
    if (tid == 0) {
      st.cand[static_cast<int64_t>(node) * a.F + f] = SmallCand{0.0, 0u, 0};
      if (!root) st.cand[static_cast<int64_t>(sib) * a.F + f] = SmallCand{0.0, 0u, 0};
    }
    return;
  }
  const int n_bins = st.counts[f], rp = st.rp[f];
  const int64_t fs = static_cast<int64_t>(a.F) * a.S;
  // sums of grads over any rows lie between -down and up, less than 2^32 apart: the lower half of a sum + down is the sum + down
  const uint32_t down  = static_cast<uint32_t>(st.q_stats[1]);
  const double down_of = static_cast<double>(down);
  const double inv_g = st.scales[2], inv_h = st.scales[3];
  const double reg   = 1e-5 > a.l2 ? 1e-5 : a.l2;
  uint2* const hist         = st.hist[p.depth & 1];
  const uint2* const parent = st.hist[(p.depth & 1) ^ 1] + static_cast<int64_t>(pair) * a.K * fs + static_cast<int64_t>(f) * a.S;
  double best_n = 0.0, best_s = 0.0;
  unsigned key_n = 0, key_s = 0;
  bool less_n = false, less_s = false;  // the best split's left child has the smaller hessian (of the first output)
  uint2 best_cell_n = make_uint2(0, 0), best_cell_s = make_uint2(0, 0);  // kLast: what lies left of it
  auto run = [&](auto plains) {
    auto quotient = [&](double grad, double hess) {
      if constexpr (decltype(plains)::value)
        return quotient_plain(grad * grad, hess + reg);
      else
        return leaf_gain_select(grad, hess, a.l1, reg);
    };
    // kAhead: the images and the parent's bin of the next output are on their way while an output's are summed
    unsigned long long ahead[kAhead > 0 ? kAhead : 1];
    uint2 parent_ahead = make_uint2(0, 0);
    const int64_t step = static_cast<int64_t>(p.built) * a.K * fs;
    auto fetch = [&](int k, int bin) {
      const int64_t at = k * fs + min(bin, max(n_bins, 1) - 1);
      const unsigned long long* const img = st.images + static_cast<int64_t>(pair) * a.K * fs + static_cast<int64_t>(f) * a.S + at;
#pragma unroll
      for (int c = 0; c < kAhead; c++) ahead[c] = img[min(c, p.chunks - 1) * step];
      if (!root) parent_ahead = parent[at];
    };
    if constexpr (kAhead > 0) fetch(0, tid);
    for (int base = 0; base < n_bins; base += kScan) {
      const int bin = base + tid;
      const bool in = bin < n_bins;
      double gain_n = 0.0, gain_s = 0.0;
      bool dead_n = !in, dead_s = !in || root;
      bool left_n = false, left_s = false;
      uint2 cell_n = make_uint2(0, 0), cell_s = make_uint2(0, 0);  // kLast
      for (int k = 0; k < a.K; k++) {
        uint32_t raw_g = 0, raw_h = 0;  // of the bin, lower halves
        uint2 pv = make_uint2(0, 0);
        I64Pair ns = st.node_sums[static_cast<int64_t>(p.level_first + node) * a.K + k];
        // (the root's, which has no sibling, are its own: behind a condition hipcc waits for them before it asks for anything else)
        I64Pair ss = st.node_sums[static_cast<int64_t>(p.level_first + (root ? node : sib)) * a.K + k];
        if constexpr (kAhead > 0) {
#pragma unroll
          for (int c = 0; c < kAhead; c++) {
            raw_g += c < p.chunks ? static_cast<uint32_t>(ahead[c] >> 32) : 0u;
            raw_h += c < p.chunks ? static_cast<uint32_t>(ahead[c]) : 0u;
          }
          pv = parent_ahead;
          const unsigned long long* const img =
            st.images + (static_cast<int64_t>(pair) * a.K + k) * fs + static_cast<int64_t>(f) * a.S + min(bin, n_bins - 1);
          for (int c = kAhead; c < p.chunks; c += kAhead) {
            unsigned long long w[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; u++) w[u] = img[min(c + u, p.chunks - 1) * step];
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
              raw_g += c + u < p.chunks ? static_cast<uint32_t>(w[u] >> 32) : 0u;
              raw_h += c + u < p.chunks ? static_cast<uint32_t>(w[u]) : 0u;
            }
          }
          raw_g = in ? raw_g : 0u;
          raw_h = in ? raw_h : 0u;
          if (k + 1 < a.K)
            fetch(k + 1, bin);
          else if (base + kScan < n_bins)
            fetch(0, bin + kScan);
        } else if (in) {
          const unsigned long long* img = st.images + (static_cast<int64_t>(pair) * a.K + k) * fs + static_cast<int64_t>(f) * a.S + bin;
          if (!root) pv = parent[k * fs + bin];
          int c = 0;
          auto add = [&](auto width) {
            constexpr int kW = decltype(width)::value;
            for (; c + kW <= p.chunks; c += kW) {
              unsigned long long w[kW];
#pragma unroll
              for (int u = 0; u < kW; u++) w[u] = img[(c + u) * step];
#pragma unroll
              for (int u = 0; u < kW; u++) {
                raw_g += static_cast<uint32_t>(w[u] >> 32);
                raw_h += static_cast<uint32_t>(w[u]);
              }
            }
          };
          add(std::integral_constant<int, 8>{});
          add(std::integral_constant<int, 1>{});
        }
        uint32_t g = wave_inclusive_sum32(raw_g);
        uint32_t h = wave_inclusive_sum32(raw_h);
        if (lane == 63) s_tot[k & 1][wave] = make_uint2(g, h);
        __syncthreads();
        if (base > 0) {
          g += s_carry[k].x;
          h += s_carry[k].y;
        }
        for (int w = 0; w < kScan / 64; w++) {
          g += w < wave ? s_tot[k & 1][w].x : 0;
          h += w < wave ? s_tot[k & 1][w].y : 0;
        }
        // the bin as it was accumulated where neither running sum is positive (build_tree.cu:645): no hessian is negative, so
        // it then has none
        const uint32_t kept = h == 0 && g + down <= down ? raw_g : g;
        // all that was asked for, before the stores below: a wait for it behind them would wait for them too (11,094 x 120, 5 outputs, 512 samples,
        // depth 8: 117 us a launch, and 101)
        arrived(ns), arrived(ss);
        asm volatile("" : "+v"(pv.x), "+v"(pv.y));
        // whole numbers below 2^35 and their differences are exact as doubles
        const double nlg = static_cast<double>(kept + down) - down_of, nlh = static_cast<double>(h);
        const double slg = static_cast<double>(pv.x + down) - down_of - nlg, slh = static_cast<double>(pv.y) - nlh;
        const double nrg = static_cast<double>(ns.grad) - nlg, nrh = static_cast<double>(ns.hess) - nlh;
        const double srg = static_cast<double>(ss.grad) - slg, srh = static_cast<double>(ss.hess) - slh;
        const double n_left = quotient(nlg * inv_g, nlh * inv_h), n_right = quotient(nrg * inv_g, nrh * inv_h);
        const double s_left = quotient(slg * inv_g, slh * inv_h), s_right = quotient(srg * inv_g, srh * inv_h);
        const double n_own = quotient(static_cast<double>(ns.grad) * inv_g, static_cast<double>(ns.hess) * inv_h);
        const double s_own = quotient(static_cast<double>(ss.grad) * inv_g, static_cast<double>(ss.hess) * inv_h);
        if (kLess && k == 0) {
          left_n = nlh < nrh;
          left_s = slh < srh;
        }
        dead_n |= nlh <= 0 || nrh <= 0;
        dead_s |= slh <= 0 || srh <= 0;
        gain_n += 0.5 * (n_left + n_right - n_own) - a.min_split_gain;
        gain_s += 0.5 * (s_left + s_right - s_own) - a.min_split_gain;
        if constexpr (kLast) {
          cell_n = make_uint2(kept, h);
          cell_s = make_uint2(pv.x - kept, pv.y - h);
        } else if (in) {
          const int64_t at = static_cast<int64_t>(k) * fs + static_cast<int64_t>(f) * a.S + bin;
          hist[static_cast<int64_t>(node) * a.K * fs + at] = make_uint2(kept, h);
          if (!root) hist[static_cast<int64_t>(sib) * a.K * fs + at] = make_uint2(pv.x - kept, pv.y - h);
        }
        // the carry of a tile is read by the next one; a barrier of the next output lies between
        if (base + kScan < n_bins) {
          __syncthreads();
          if (tid == kScan - 1) s_carry[k] = make_uint2(g, h);
        }
      }
      const unsigned key = tie_key_of_bin(rp + bin);
      const bool take_n = !dead_n && gain_n > 0 && (gain_n > best_n || (gain_n == best_n && key > key_n));
      const bool take_s = !dead_s && gain_s > 0 && (gain_s > best_s || (gain_s == best_s && key > key_s));
      best_n = take_n ? gain_n : best_n;
      key_n  = take_n ? key : key_n;
      if constexpr (kLess) less_n = take_n ? left_n : less_n;
      if constexpr (kLast) best_cell_n = make_uint2(take_n ? cell_n.x : best_cell_n.x, take_n ? cell_n.y : best_cell_n.y);
      best_s = take_s ? gain_s : best_s;
      key_s  = take_s ? key : key_s;
      if constexpr (kLess) less_s = take_s ? left_s : less_s;
      if constexpr (kLast) best_cell_s = make_uint2(take_s ? cell_s.x : best_cell_s.x, take_s ? cell_s.y : best_cell_s.y);
      if (base + kScan < n_bins) __syncthreads();
    }
  };
  if (plain_quotients(a.l1, inv_g, inv_h, reg))
    run(std::true_type{});
  else
    run(std::false_type{});
  const double own_n = best_n, own_s = best_s;
  const unsigned own_key_n = key_n, own_key_s = key_s;
  wave_best_key(best_n, key_n);
  wave_best_key(best_s, key_s);
  if constexpr (kLess) {
    less_n = __any(less_n && own_key_n == key_n && own_n == best_n);  // (no two lanes have one key)
    less_s = __any(less_s && own_key_s == key_s && own_s == best_s);
  }
  if constexpr (kLast) {
    if (key_n != 0 && own_key_n == key_n && own_n == best_n) s_cell[0][wave] = best_cell_n;
    if (key_s != 0 && own_key_s == key_s && own_s == best_s) s_cell[1][wave] = best_cell_s;
  }
  if (lane == 0) {
    s_best[0][wave] = best_n;
    s_bkey[0][wave] = key_n;
    s_less[0][wave] = less_n ? kLeftSmaller : 0;
    s_best[1][wave] = best_s;
    s_bkey[1][wave] = key_s;
    s_less[1][wave] = less_s ? kLeftSmaller : 0;
  }
  __syncthreads();
  if (tid < (root ? 1 : 2)) {
    double best  = 0.0;
    unsigned key = 0;
    int less     = 0, from = 0;
    for (int w = 0; w < kScan / 64; w++) {
      const bool take = s_best[tid][w] > best || (s_best[tid][w] == best && s_bkey[tid][w] > key);
      best = take ? s_best[tid][w] : best;
      key  = take ? s_bkey[tid][w] : key;
      less = take ? s_less[tid][w] : less;
      from = take ? w : from;
    }
    if (kLast && key != 0) st.left[static_cast<int64_t>(tid == 0 ? node : sib) * a.F + f] = s_cell[tid][from];
    st.cand[static_cast<int64_t>(tid == 0 ? node : sib) * a.F + f] = SmallCand{best, key, key != 0 ? (bin_of_tie_key(key) - rp) | less : 0};
  }
}

// The same with a wave for a (pair of siblings, feature), 64 bins at a time: no barrier, no exchange through the LDS, and the terms that do not
// depend on the bin once an output instead of once a thread. Below the root, where nobody asks for the smaller child, and from kWavePairs on:
// with fewer the waves of a workgroup, which take the bins of a feature at a time, finish sooner than one that takes them in turn (50,000 x 200,
// 256 samples, levels of 1600, 3200, 6400 and 12,800 pairs and features: 8.8, 12.2, 18.0 and 27.7 us, by workgroups with 16 bytes a bin 13.6, 19.4,
// 33.1 and 61.2. As the bound 512 gives scans of 90 us a tree for 85 with 30,000 x 60 and 8 outputs, 98 for 103 with 50,000 x 100 and 2, 2048 86
// and 111.) A tree of 50,000 x 200, depth 8: 353 us, now 297; of 20,000 x 60, 128 samples, depth 10, 351 and 306; of 50,000 x 100 with 2 outputs, 64
// samples, depth 9, 405 and 319.
template <bool kLast>
__global__ void __launch_bounds__(kScan)
  mid_scan_waves_kernel(MidArgs a, MidTreeState st, LevelPlan p)
{
  const int lane = threadIdx.x & 63;
  const int item = static_cast<int>(blockIdx.x) * (kScan / 64) + __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int f = item % a.F, pair = item / a.F;
  if (pair >= p.built || level_is_empty(st, p.depth)) return;
  const I64Pair* const sums = st.node_sums + static_cast<int64_t>(p.level_first + 2 * pair) * a.K;  // the left child's, then the right one's
  const int64_t left_h = sums[0].hess, right_h = sums[a.K].hess;
  // the children of a node that did not split have no rows
  if (left_h <= 0) return;
  const int own = left_h < right_h ? 0 : 1;  // built_of_pair
  const int64_t node = 2 * pair + own, sib = node ^ 1;
  if (a.feature_set != nullptr && a.feature_set[f] == 0) {
    if (lane < 2) st.cand[(2 * pair + lane) * static_cast<int64_t>(a.F) + f] = SmallCand{0.0, 0u, 0};
    return;
  }
  const int n_bins = st.counts[f], rp = st.rp[f];
  const int64_t fs = static_cast<int64_t>(a.F) * a.S;
  const uint32_t down  = static_cast<uint32_t>(st.q_stats[1]);
  const double down_of = static_cast<double>(down);
  const double inv_g = st.scales[2], inv_h = st.scales[3];
  const double reg   = 1e-5 > a.l2 ? 1e-5 : a.l2;
  uint2* const hist         = st.hist[p.depth & 1];
  const uint2* const parent = st.hist[(p.depth & 1) ^ 1] + static_cast<int64_t>(pair) * a.K * fs + static_cast<int64_t>(f) * a.S;
  const unsigned long long* const images = st.images + static_cast<int64_t>(pair) * a.K * fs + static_cast<int64_t>(f) * a.S;
  const int64_t step = static_cast<int64_t>(p.built) * a.K * fs;
  // lane k: sums of output k, and the term of the gains that does not depend on the bin
  I64Pair ns{0, 0}, ss{0, 0};
  if (lane < a.K) {
    ns = sums[own * a.K + lane];
    ss = sums[(own ^ 1) * a.K + lane];
  }
  const double all_ng = static_cast<double>(ns.grad), all_nh = static_cast<double>(ns.hess);
  const double all_sg = static_cast<double>(ss.grad), all_sh = static_cast<double>(ss.hess);
  double best_n = 0.0, best_s = 0.0;
  unsigned key_n = 0, key_s = 0;
  uint2 best_cell_n = make_uint2(0, 0), best_cell_s = make_uint2(0, 0);  // kLast: what lies left of it
  auto run = [&](auto plains) {
    auto quotient = [&](double grad, double hess) {
      if constexpr (decltype(plains)::value)
        return quotient_plain(grad * grad, hess + reg);
      else
        return leaf_gain_select(grad, hess, a.l1, reg);
    };
    const double own_n = quotient(all_ng * inv_g, all_nh * inv_h), own_s = quotient(all_sg * inv_g, all_sh * inv_h);
    // the images and the parent's bins of the next 64 bins (or of the next output's) are on their way while these are summed
    constexpr int kAhead = 4;
    unsigned long long ahead[kAhead];
    uint2 parent_ahead;
    const int tiles = (n_bins + 63) / 64, items = tiles * a.K;
    int next_k = 0, next_bin = lane;
    auto fetch = [&]() {
      const int64_t at = next_k * fs + min(next_bin, max(n_bins, 1) - 1);
#pragma unroll
      for (int c = 0; c < kAhead; c++) ahead[c] = images[at + min(c, p.chunks - 1) * step];
      parent_ahead = parent[at];
      if (++next_k == a.K) {
        next_k = 0;
        next_bin += 64;
      }
    };
    fetch();
    uint32_t agg_g = 0, agg_h = 0;  // lane k: output k's sums of the bins so far
    int k = 0, bin = lane;
    double gain_n = 0.0, gain_s = 0.0;
    bool live_n = true, live_s = true;
    for (int i = 0; i < items; i++) {
      const bool in = bin < n_bins;
      uint32_t raw_g = 0, raw_h = 0;
#pragma unroll
      for (int c = 0; c < kAhead; c++) {
        raw_g += c < p.chunks ? static_cast<uint32_t>(ahead[c] >> 32) : 0u;
        raw_h += c < p.chunks ? static_cast<uint32_t>(ahead[c]) : 0u;
      }
      const uint2 pv     = parent_ahead;
      const int64_t here = k * fs + min(bin, n_bins - 1);
      for (int c = kAhead; c < p.chunks; c += 4) {
        unsigned long long w[4];
#pragma unroll
        for (int u = 0; u < 4; u++) w[u] = images[here + min(c + u, p.chunks - 1) * step];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          raw_g += c + u < p.chunks ? static_cast<uint32_t>(w[u] >> 32) : 0u;
          raw_h += c + u < p.chunks ? static_cast<uint32_t>(w[u]) : 0u;
        }
      }
      if (i + 1 < items) fetch();
      raw_g = in ? raw_g : 0u;
      raw_h = in ? raw_h : 0u;
      const uint32_t g = wave_inclusive_sum32(raw_g) + wave_read_lane32(agg_g, k);
      const uint32_t h = wave_inclusive_sum32(raw_h) + wave_read_lane32(agg_h, k);
      const uint32_t to_g = wave_read_lane32(g, 63), to_h = wave_read_lane32(h, 63);
      if (lane == k) {
        agg_g = to_g;
        agg_h = to_h;
      }
      // (the rule on bins that the reference leaves as they are, see mid_scan_kernel)
      const uint32_t kept = h == 0 && g + down <= down ? raw_g : g;
      const double nlg = static_cast<double>(kept + down) - down_of, nlh = static_cast<double>(h);
      const double slg = static_cast<double>(pv.x + down) - down_of - nlg, slh = static_cast<double>(pv.y) - nlh;
      const double nrg = wave_read_lane_f64(all_ng, k) - nlg, nrh = wave_read_lane_f64(all_nh, k) - nlh;
      const double srg = wave_read_lane_f64(all_sg, k) - slg, srh = wave_read_lane_f64(all_sh, k) - slh;
      const double n_left = quotient(nlg * inv_g, nlh * inv_h), n_right = quotient(nrg * inv_g, nrh * inv_h);
      const double s_left = quotient(slg * inv_g, slh * inv_h), s_right = quotient(srg * inv_g, srh * inv_h);
      live_n = live_n && nlh > 0 && nrh > 0;
      live_s = live_s && slh > 0 && srh > 0;
      gain_n += 0.5 * (n_left + n_right - wave_read_lane_f64(own_n, k)) - a.min_split_gain;
      gain_s += 0.5 * (s_left + s_right - wave_read_lane_f64(own_s, k)) - a.min_split_gain;
      if (!kLast && in) {
        hist[node * a.K * fs + static_cast<int64_t>(f) * a.S + here] = make_uint2(kept, h);
        hist[sib * a.K * fs + static_cast<int64_t>(f) * a.S + here]  = make_uint2(pv.x - kept, pv.y - h);
      }
      if (++k == a.K) {
        const unsigned key = tie_key_of_bin(rp + bin);
        const bool take_n = in && live_n && gain_n > 0 && (gain_n > best_n || (gain_n == best_n && key > key_n));
        const bool take_s = in && live_s && gain_s > 0 && (gain_s > best_s || (gain_s == best_s && key > key_s));
        best_n = take_n ? gain_n : best_n;
        key_n  = take_n ? key : key_n;
        best_s = take_s ? gain_s : best_s;
        key_s  = take_s ? key : key_s;
        if constexpr (kLast) {
          best_cell_n = make_uint2(take_n ? kept : best_cell_n.x, take_n ? h : best_cell_n.y);
          best_cell_s = make_uint2(take_s ? pv.x - kept : best_cell_s.x, take_s ? pv.y - h : best_cell_s.y);
        }
        k = 0;
        bin += 64;
        gain_n = gain_s = 0.0;
        live_n = live_s = true;
      }
    }
  };
  if (plain_quotients(a.l1, inv_g, inv_h, reg))
    run(std::true_type{});
  else
    run(std::false_type{});
  const double lane_n = best_n, lane_s = best_s;
  const unsigned lane_key_n = key_n, lane_key_s = key_s;
  wave_best_key(best_n, key_n);
  wave_best_key(best_s, key_s);
  if constexpr (kLast) {
    // (no two lanes have one key)
    if (key_n != 0 && lane_key_n == key_n && lane_n == best_n) st.left[node * a.F + f] = best_cell_n;
    if (key_s != 0 && lane_key_s == key_s && lane_s == best_s) st.left[sib * a.F + f] = best_cell_s;
  }
  if (lane < 2) {
    const unsigned key = lane == 0 ? key_n : key_s;
    st.cand[(lane == 0 ? node : sib) * a.F + f] = SmallCand{lane == 0 ? best_n : best_s, key, key != 0 ? bin_of_tie_key(key) - rp : 0};
  }
}

// Splits of a level of many nodes, one group of lanes per node.
__global__ void __launch_bounds__(kScan)
  mid_decide_kernel(MidArgs a, MidTreeState st, LevelPlan p, int lanes_log)
{
  if (level_is_empty(st, p.depth)) return;
  const int lanes = 1 << lanes_log, sub = threadIdx.x & (lanes - 1);
  const int j     = (blockIdx.x * kScan + static_cast<int>(threadIdx.x)) >> lanes_log;
  const int2 sp   = decide_node(a, st, p, j < p.n_nodes ? j : -1, sub, lanes, true);
  if (sub == 0 && j < p.n_nodes) st.splits[j] = sp;
}

// kDecided: mid_decide_kernel has run; otherwise every workgroup finds the splits for itself (few nodes: it
// saves a launch) and the nodes' outputs are dealt to the workgroups.
template <typename BinT, bool kDecided>
__global__ void __launch_bounds__(kWide)
  mid_apply_kernel(MidArgs a, MidTreeState st, LevelPlan p, int lanes_log, uint16_t* row_node)
{
  __shared__ int2 s_split[kMidMaxLevelNodes];
  const int tid = threadIdx.x;
  const int r   = blockIdx.x * kRowsApply + 4 * tid;
  uint2 nd      = make_uint2(0xffffffffu, 0xffffffffu);
  if (r < a.N) nd = *reinterpret_cast<const uint2*>(row_node + r);
  if (level_is_empty(st, p.depth)) return;
  if constexpr (kDecided) {
    for (int j = tid; j < p.n_nodes; j += kWide) s_split[j] = st.splits[j];
  } else {
    const int lanes = 1 << lanes_log, sub = tid & (lanes - 1);
    for (int j0 = 0; j0 < p.n_nodes; j0 += kWide >> lanes_log) {
      const int j   = j0 + (tid >> lanes_log);
      const int2 sp = decide_node(a, st, p, j < p.n_nodes ? j : -1, sub, lanes,
                                  j % static_cast<int>(gridDim.x) == static_cast<int>(blockIdx.x));
      if (sub == 0 && j < p.n_nodes) s_split[j] = sp;
    }
  }
  __syncthreads();
  if (r >= a.N) return;
  const unsigned node[4] = {nd.x & 0xffffu, nd.x >> 16, nd.y & 0xffffu, nd.y >> 16};
  const RowSplits<BinT> rows(a, st, s_split, node, r);
  rows.store_leaves(a, p, node, r, p.last);
  if (!p.last)
    *reinterpret_cast<uint2*>(row_node + r) = make_uint2(rows.next[0] | rows.next[1] << 16, rows.next[2] | rows.next[3] << 16);
}

// For the profiler: the rows of the level's nodes and of those that are accumulated.
__global__ void __launch_bounds__(kScan) mid_count_kernel(MidArgs a, MidTreeState st, LevelPlan p, const uint16_t* row_node,
                                                         LevelMeta* total)
{
  const int r    = blockIdx.x * kScan + threadIdx.x;
  const int node = r < a.N ? row_node[r] : kNone;
  const bool has = node != kNone && !level_is_empty(st, p.depth);
  const bool built = has && (p.depth == 0 || built_of_pair(st.node_sums, p.level_first, node >> 1, a.K) == node);
  const unsigned long long all = __ballot(has), some = __ballot(built);
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(reinterpret_cast<unsigned long long*>(&total->instances), static_cast<unsigned long long>(__popcll(all)));
    atomicAdd(reinterpret_cast<unsigned long long*>(&total->built_instances), static_cast<unsigned long long>(__popcll(some)));
  }
  if (r < p.built && (p.depth == 0 || st.node_sums[static_cast<int64_t>(p.level_first + 2 * r) * a.K].hess > 0))
    atomicAdd(reinterpret_cast<unsigned long long*>(&total->built_nodes), 1ULL);
}

// One level's plan. A workgroup of the histogram pass keeps fw features of bw nodes in the LDS; near the root
// several features share the loads of a row, deeper a feature's nodes fill the LDS and then come in
// blocks. Ranges of rows are cut until there is a workgroup for every CU or so, not below 3072 rows (1024 up to
// 16 ranges), and only so many that their images (written here, read by the scan) stay within 64 MB (one always).
LevelPlan plan_level(int64_t N, int F, int K, int S, int depth, int max_depth)
{
  LevelPlan p;
  p.depth       = depth;
  p.level_first = static_cast<int>(level_begin(depth));
  p.n_nodes     = 1 << depth;
  p.built       = depth == 0 ? 1 : p.n_nodes / 2;
  p.last        = depth + 1 == max_depth;
  const int rows_of_lds = std::max<int>(1, static_cast<int>(kHistLds / (static_cast<size_t>(S) * 8)));
  const bool by_images = N * F * K <= kImageValues;
  p.fw   = std::max(1, std::min({rows_of_lds / p.built, by_images && K == 1 ? 2 : kMaxFw, F}));
  p.bw   = std::max(1, std::min(p.built, rows_of_lds / p.fw));
  p.n_fb = (F + p.fw - 1) / p.fw;
  p.n_bb = (p.built + p.bw - 1) / p.bw;
  const int64_t inner = static_cast<int64_t>(p.n_fb) * p.n_bb * K;
  const int64_t image = static_cast<int64_t>(p.built) * K * F * S * 8;
  // Two workgroups share a CU where their histograms do. By images too where only that leaves the eight ranges that the
  // XCDs take one each (several outputs: 50,000 x 20 with 8, depth 6, 278 us a tree with six ranges, 258 with eight; 20,000 x 10
  // with 16 361 and 318): with fewer, whichever it is, the images count more (30,000 x 25 with 16 outputs 335 with two, 378 with four).
  const bool too_few  = K > 1 && 256 / inner < 8 && 512 / inner >= 8;
  p.pairs             = (!by_images || too_few) && static_cast<size_t>(p.fw) * p.bw * S * 8 <= 72 * 1024;
  int64_t chunks      = std::max<int64_t>(1, (p.pairs ? 512 : 256) / inner);
  // (three quarters of a workgroup's threads have rows: with 1024 rows a range, most of them had none and the scan
  // added up twice the images: 100,000 x 32, 10 rounds, 2.06 -> 1.87 ms; 60,000 x 20 with 4 outputs -9 %)
  chunks              = std::min(chunks, std::max<int64_t>({1, N / 3072, std::min<int64_t>(16, N / 1024)}));
  chunks              = std::min<int64_t>(chunks, 64);
  chunks              = std::min(chunks, std::max<int64_t>(1, (int64_t(64) << 20) / image));
  if (chunks > 8) chunks = chunks / 8 * 8;
  // Few rows: the images are then far larger than the rows (64 ranges of 100,000 x 32 at depth 5: 67 MB written and
  // read again for 3 MB of bins). Fewer ranges, and blocks of fewer nodes to keep as many workgroups, as
  // long as a workgroup's rows take it no more than two passes: that level 31.3 -> 22.4 us (histogram and scan).
  while (p.bw >= 2 && chunks >= 16 && chunks * image > (int64_t(8) << 20) && (N + chunks / 2 - 1) / (chunks / 2) <= 8192) {
    chunks /= 2;
    p.bw   = (p.bw + 1) / 2;
    p.n_bb = (p.built + p.bw - 1) / p.bw;
  }
  p.chunks     = static_cast<int>(chunks);
  p.chunk_rows = static_cast<int>(((N + chunks - 1) / chunks + 3) / 4 * 4);
  return p;
}

}  // namespace

// Scanned histograms of two levels and the images of the level that has most of them.
size_t mid_hist_bytes(int64_t N, int F, int K, int max_depth, int S)
{
  const int64_t fs = static_cast<int64_t>(K) * F * S;
  int64_t images   = 0;
  for (int d = 0; d < max_depth; d++) {
    const LevelPlan p = plan_level(N, F, K, S, d, max_depth);
    images            = std::max(images, static_cast<int64_t>(p.chunks) * p.built * fs);
  }
  return static_cast<size_t>(2 * (int64_t(1) << (max_depth - 1)) * fs) * sizeof(uint2) + static_cast<size_t>(images) * 8;
}

// By size: measured against the general builder (one output, depth 8 and 256 samples unless stated), us: 20,000 x 100
// 470 -> 191 at depth 6, 250,000 x 43 764 -> 323, 500,000 x 50 849 -> 396, 1,000,000 x 30 955 -> 399, 2,000,000 x 40
// 1139 -> 763, 600,000 x 50 with 8 outputs 1652 -> 1511, 2,000,000 x 80 1398 -> 1133. Every pass reads all rows, and
// where a level's nodes come in several blocks once per block (800,000 x 40 with 512 samples at depth 10, eight
// blocks: 1323 -> 1231), so what counts is values times blocks of the last level: at 240 million the two are about
// even (6,000,000 x 40 2034 -> 1955, 800,000 x 300 1952 -> 1913, 3,000,000 x 80 1752 -> 1672).
bool mid_tree_fits(int64_t N, int F, int K, int max_depth, int S)
{
  if (max_depth < 1 || max_depth > kMidMaxDepth || K > kMidMaxOutputs || S > LBT_MAX_SPLIT_SAMPLES) return false;
  // the chunk sums are added up by one workgroup, bins numbered with 26 bits (tie_key_of_bin), rows with 31
  if (N * K > int64_t(4096) * 4096 || static_cast<int64_t>(F) * S >= (int64_t(1) << 26)) return false;
  const int64_t level_hist = (int64_t(1) << (max_depth - 1)) * K * F * S * 16;
  if (level_hist > (int64_t(768) << 20)) return false;
  const int64_t values = N * F * K;
  return values * plan_level(N, F, K, S, max_depth - 1, max_depth).n_bb <= kMidMaxValues;
}

// Of two builders that both could, the one for few rows or this one. A level costs the first less to begin with and
// more per entry (one workgroup per feature walks them in order, output by output); here it is the histograms that
// count, and a scan workgroup per node and feature. The two sums are times of a tree in us, fitted to 190 shapes (300
// to 8192 rows, 3 to 500 features, 1 to 16 outputs, depth 2 to 10, 64 to 1024 samples, float and double) when both
// builders took a launch more per level, with 15 % in favour of the first. Of 260 shapes timed again with the present kernels (1000 to 8192 rows,
// 8 to 250 features, 1 and 4 outputs, depth 4 to 10) none where this builder is taken is slower for it; 34 where the first one is taken would be 4 to
// 39 % faster here, most of them one output of 4500 to 6500 rows and up to 60 features: the line lies too high there. Both now, few rows
// against medium: 8 features, depth 8 at 1000, 4096 and 8192 rows 83, 122, 209 and 135, 146, 145; 5000 x 8, depth 6 140 and 105; 8192 x 20,
// depth 6 168 and 110; 20 features, 4 outputs, depth 6 at 1000, 2000 and 8192 rows 123, 154, 437 and 131, 134, 151; 8192 x 250 with 4, depth 8
// 686 and 591.
bool mid_beats_small(int64_t N, int F, int K, int max_depth, int S)
{
  const double d = max_depth, n = static_cast<double>(N), f = F, k = K;
  const double small_us = 25.0 + d * (8.7 + 2.0 * k + 1.8e-3 * n * k * (N > 4096 && K > 1 ? 1.5 : 1.0) + 7.1e-6 * n * f);
  const double nodes = static_cast<double>(int64_t(1) << max_depth), tiles = (S + kScan - 1) / kScan;
  // histograms of all nodes in MB, or of those that rows reach: four bins per value and level (16 bytes a bin, as the sum was fitted; they take 8 now)
  const double hist_mb = std::min(nodes * f * S * k * 16.0, n * f * k * d * 64.0) / 1048576.0;
  const double mid_us  = 16.0 + d * (19.5 + 1.14 * k * tiles) + 0.29 * hist_mb + 1.0e-3 * nodes * f * k * tiles + 1.74e-6 * n * f * k * d;
  return 1.15 * mid_us < small_us;
}

// Whether the workgroups of level p's histograms find the nodes of their rows for themselves, which saves the launch that does.
// All workgroups of a range of rows do so for the same rows, a byte gathered per row and workgroup: up to 2.5 million
// such visits it pays. Trees with the launch and without, us: 78,125 x 64, depth 6 (2.5 million) 167 and 155; 100,000 x 32, depth 6 162
// and 151; 60,000 x 20 with 4 outputs, depth 6 197 and 184; 400,000 x 12, depth 6 169 and 156. By one workgroup of two features to a CU
// it still gains 3 % at 4 million and nothing at 6; with four features 800,000 x 16, depth 8 (3.2 million) takes 287 and 291, 1,000,000 x
// 30 with 8 million 3 % more. Where two workgroups share a CU, half as many: with 8 outputs, depth 6 and 8, 20,000 x 20 (0.8 million)
// 251 and 245, 343 and 334; 35,000 x 20 (1.4 million) 256 and 258, 350 and 354; 62,000 x 20 266 and 270, 365 and 371. And where they
// are no more than the CUs: those that wait for a CU decide all over again (depth 5: 9000 x 500, 250 workgroups, 181 and 170, 6000 x 500 with
// 2 outputs, 250, 206 and 194; 6500 x 700, 350, 219 and 224, 6000 x 500 with 3, 375, 244 and 249).
static bool nodes_with_histograms(const MidArgs& a, const LevelPlan& p)
{
  const int64_t inner = static_cast<int64_t>(p.n_fb) * p.n_bb * a.K;  // workgroups of a range of rows
  return p.depth > 0 && inner <= 256 && inner * a.N <= (p.pairs ? kNodesMost / 2 : kNodesMost);
}

template <typename BinT, Nodes kNodes>
static int launch_histograms(hipStream_t stream, const MidTreeState& st, const MidArgs& a, const LevelPlan& p, const LevelPlan& above,
                             int lanes_log, const uint16_t* from, uint16_t* to)
{
  ProfScope ps(LBT_PROF_HISTOGRAM, stream, 0.0, p.depth);
  static std::atomic<bool> attr_set[kMaxDevices] = {};
  LBT_TRY((allow_dynamic_lds(mid_histogram_kernel<BinT, kNodes>, kHistLds + 4096, attr_set)));
  const int lanes8    = p.chunks >= 8 ? 8 : 1;
  const int writers   = kNodes == Nodes::kDecide ? ((above.n_nodes << lanes_log) + kWide - 1) / kWide : 0;
  const unsigned grid = static_cast<unsigned>((p.chunks + lanes8 - 1) / lanes8 * lanes8 * p.n_fb * p.n_bb * a.K + writers);
  mid_histogram_kernel<BinT, kNodes><<<grid, kWide, static_cast<size_t>(p.fw) * p.bw * a.S * 8, stream>>>(
    a, st, p, above, lanes_log, writers, from, to);
  return LBT_OK;
}

template <bool kLess>
static auto scan_of(int K, int chunks)
{
  if (K == 1) return mid_scan_kernel<kLess, false, 0>;
  return chunks <= 4 ? mid_scan_kernel<kLess, false, 4> : chunks <= 8 ? mid_scan_kernel<kLess, false, 8> : mid_scan_kernel<kLess, false, 16>;
}

template <typename T, typename BinT>
static int queue_levels(hipStream_t stream, const MidTreeState& st, const MidArgs& a, const DeviceAnswer& answer,
                        LevelMeta* level_totals)
{
  int lanes_log = 0;
  while (lanes_log < 6 && (1 << lanes_log) < a.F) lanes_log++;
  int cur    = 0;                     // row_node[cur] holds the rows' nodes of the level, or of the one above it
  Nodes how  = Nodes::kCarried;
  LevelPlan above{};
  for (int d = 0; d < a.max_depth && (d == 0 || !answer.declined()); d++) {
    const LevelPlan p = plan_level(a.N, a.F, a.K, a.S, d, a.max_depth);
    const uint16_t* const from = st.row_node[cur];
    uint16_t* const to         = st.row_node[cur ^ 1];
    const bool later           = !p.last && nodes_with_histograms(a, plan_level(a.N, a.F, a.K, a.S, d + 1, a.max_depth));
    switch (how) {
      case Nodes::kCarried: LBT_TRY((launch_histograms<BinT, Nodes::kCarried>(stream, st, a, p, above, lanes_log, from, nullptr))); break;
      case Nodes::kDecide: LBT_TRY((launch_histograms<BinT, Nodes::kDecide>(stream, st, a, p, above, lanes_log, from, to))); break;
      case Nodes::kDecided: LBT_TRY((launch_histograms<BinT, Nodes::kDecided>(stream, st, a, p, above, lanes_log, from, to))); break;
    }
    if (how != Nodes::kCarried) cur ^= 1;
    if (level_totals != nullptr)
      mid_count_kernel<<<static_cast<unsigned>((a.N + kScan - 1) / kScan), kScan, 0, stream>>>(a, st, p, st.row_node[cur], level_totals + d);
    {
      ProfScope ps(LBT_PROF_SCAN, stream);
      const unsigned grid = static_cast<unsigned>(p.built) * a.F;
      if (later)
        scan_of<true>(a.K, p.chunks)<<<grid, kScan, 0, stream>>>(a, st, p);
      else if (d > 0 && static_cast<int64_t>(grid) >= kWavePairs && p.last && a.K == 1)
        mid_scan_waves_kernel<true><<<(grid + kScan / 64 - 1) / (kScan / 64), kScan, 0, stream>>>(a, st, p);
      else if (d > 0 && static_cast<int64_t>(grid) >= kWavePairs)
        mid_scan_waves_kernel<false><<<(grid + kScan / 64 - 1) / (kScan / 64), kScan, 0, stream>>>(a, st, p);
      else if (p.last && a.K == 1)
        mid_scan_kernel<false, true, 0><<<grid, kScan, 0, stream>>>(a, st, p);
      else
        scan_of<false>(a.K, p.chunks)<<<grid, kScan, 0, stream>>>(a, st, p);
    }
    ProfScope ps(LBT_PROF_POSITIONS, stream);
    const unsigned grid = static_cast<unsigned>((a.N + kRowsApply - 1) / kRowsApply);
    // few nodes: every workgroup that asks for the splits finds them for itself (it saves a launch)
    const bool few = p.n_nodes <= 2 * (kWide >> lanes_log);
    if (!few || (later && static_cast<int64_t>(p.n_nodes) * a.F > kCandsMost)) {
      mid_decide_kernel<<<((p.n_nodes << lanes_log) + kScan - 1) / kScan, kScan, 0, stream>>>(a, st, p, lanes_log);
      how = Nodes::kDecided;
    } else {
      how = Nodes::kDecide;
    }
    above = p;
    if (later) continue;
    if (how == Nodes::kDecide)
      mid_apply_kernel<BinT, false><<<grid, kWide, 0, stream>>>(a, st, p, lanes_log, st.row_node[cur]);
    else
      mid_apply_kernel<BinT, true><<<grid, kWide, 0, stream>>>(a, st, p, lanes_log, st.row_node[cur]);
    how = Nodes::kCarried;
  }
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

template <typename T>
int mid_tree_build(hipStream_t stream, const MidTreeState& st, const T* X, int64_t row_offset, int64_t N, int F, int K,
                   const double* g, const double* h, const uint8_t* feature_set, const lbt_build_params& prm,
                   double* leaf, int32_t* feature, double* split, double* gain, double* hessian, int32_t* row_leaf,
                   int32_t* n_bins, LevelMeta* level_totals, bool* taken)
{
  *taken = false;
  DeviceAnswer answer;
  LBT_TRY(answer.open(stream));
  MidArgs a;
  a.N = static_cast<int>(N); a.F = F; a.K = K; a.S = prm.split_samples;
  a.row_offset = row_offset; a.seed = prm.seed; a.dataset_rows = prm.dataset_rows;
  a.g = g; a.h = h;
  a.m       = static_cast<int>((N * K + 4095) / 4096);
  a.chunk_a = prm.abs_sum_chunks != nullptr ? prm.abs_sum_chunks : st.chunk_sums;
  a.chunk_b = a.chunk_a + a.m;
  a.feature_set = feature_set;
  a.l1 = prm.l1_regularization; a.l2 = prm.l2_regularization; a.min_split_gain = prm.min_split_gain;
  a.max_nodes = prm.max_nodes; a.max_depth = prm.max_depth;
  // every level's histograms within the reference's buffer, whatever the number of bins (see final_histogram_range)
  const double buffer = prm.hist_cache_bytes > 0 ? static_cast<double>(prm.hist_cache_bytes) : 1e9;
  a.zeros_kept        = static_cast<double>(level_end(prm.max_depth - 1)) * K * F * a.S * 16.0 <= buffer;
  a.leaf = leaf; a.feature = feature; a.split = split; a.gain = gain; a.hessian = hessian; a.row_leaf = row_leaf;
  a.answer = answer.words; a.tag = answer.tag;
  int P = 1;
  while (P < a.S) P <<= 1;
  {
    ProfScope ps(LBT_PROF_PROPOSALS, stream);
    static std::atomic<bool> attr_set[kMaxDevices] = {};
    LBT_TRY(allow_dynamic_lds(mid_prologue_kernel<T>, 64 * 1024, attr_set));
    const int sum_groups  = prm.abs_sum_chunks != nullptr ? 0 : (a.m + 3) / 4;
    const int64_t clear   = std::max<int64_t>(static_cast<int64_t>(prm.max_nodes) * K, st.pitch / 4);
    const int clearers    = static_cast<int>(std::min<int64_t>((clear + kWide - 1) / kWide, 128));
    const size_t lds      = std::max<size_t>(static_cast<size_t>(P) * kProposalScratch<T>, 2 * kWide * sizeof(double));
    mid_prologue_kernel<T><<<F + sum_groups + clearers, kWide, lds, stream>>>(X, a, st, P, sum_groups);
  }
  {
    ProfScope ps(LBT_PROF_BINNING, stream);
    BinPlan p;
    // few entries a thread: the launch lasts as long as the quantiser's chain of loads, roundings and sums (8192 a workgroup:
    // 18 us on 100,000 x 32, whatever the binning took)
    p.quant_per    = static_cast<int>(std::min<int64_t>(8, std::max<int64_t>(1, (N * K + 128 * kWide - 1) / (128 * kWide)))) * kWide;
    p.quant_groups = static_cast<int>((N * K + p.quant_per - 1) / p.quant_per);
    p.search_steps = 0;
    while ((1 << p.search_steps) < a.S + 1) p.search_steps++;
    // features of a workgroup: what the search needs of them fits 64 KB, two workgroups a CU
    const size_t per_feature = prop_pitch(a.S) * sizeof(T) + (st.cells / kCellsPerEntry + 1) * sizeof(uint2) + 4 + (kRowsBin + 4) * st.bin_bytes;
    p.fb     = std::max(1, std::min<int>(F, std::min<int>(kMaxFb<T>, static_cast<int>(64 * 1024 / per_feature))));
    p.n_fb   = (F + p.fb - 1) / p.fb;
    p.fb     = (F + p.n_fb - 1) / p.n_fb;  // blocks of even width
    p.fb_log = 0;
    while ((1 << p.fb_log) < p.fb) p.fb_log++;
    const int tiles = static_cast<int>((N + kRowsBin - 1) / kRowsBin);
    // Tiles in equal shares to no more workgroups than run at once, two to a CU (with a few more than that the last ones take all of a second
    // turn: 250,000 x 43 in 77 us for 29): beside the quantiser's, or behind them, whichever ends sooner by some 4 us a tile and 2 us
    // for 1024 entries.
    auto tiles_each = [&](int beside) { const int most = std::max(1, (512 - beside) / p.n_fb); return (tiles + most - 1) / most; };
    const int beside = tiles_each(std::min(384, p.quant_groups)), behind = tiles_each(0);
    const int each   = 4 * beside <= 4 * behind + 4 + 2 * (p.quant_per / kWide) ? beside : behind;
    p.row_groups     = (tiles + each - 1) / each;
    const size_t lds = std::max<size_t>(static_cast<size_t>(p.fb) * per_feature + 16, 2 * kWide * sizeof(double));
    static std::atomic<bool> attr_set[2][kMaxDevices] = {};
    const unsigned grid = static_cast<unsigned>(p.quant_groups + p.n_fb * p.row_groups);
    if (st.bin_bytes == 1) {
      LBT_TRY((allow_dynamic_lds(mid_bin_kernel<T, uint8_t>, 80 * 1024, attr_set[0])));
      mid_bin_kernel<T, uint8_t><<<grid, kWide, lds, stream>>>(X, a, st, p);
    } else {
      LBT_TRY((allow_dynamic_lds(mid_bin_kernel<T, uint16_t>, 80 * 1024, attr_set[1])));
      mid_bin_kernel<T, uint16_t><<<grid, kWide, lds, stream>>>(X, a, st, p);
    }
  }
  if (st.bin_bytes == 1)
    LBT_TRY((queue_levels<T, uint8_t>(stream, st, a, answer, level_totals)));
  else
    LBT_TRY((queue_levels<T, uint16_t>(stream, st, a, answer, level_totals)));
  unsigned flags = 0;
  LBT_TRY(answer.wait(&flags, n_bins));
  *taken = flags == 0;
  return LBT_OK;
}

template int mid_tree_build<float>(hipStream_t, const MidTreeState&, const float*, int64_t, int64_t, int, int,
                                   const double*, const double*, const uint8_t*, const lbt_build_params&, double*,
                                   int32_t*, double*, double*, double*, int32_t*, int32_t*, LevelMeta*, bool*);
template int mid_tree_build<double>(hipStream_t, const MidTreeState&, const double*, int64_t, int64_t, int, int,
                                    const double*, const double*, const uint8_t*, const lbt_build_params&, double*,
                                    int32_t*, double*, double*, double*, int32_t*, int32_t*, LevelMeta*, bool*);

}  // namespace lbt
