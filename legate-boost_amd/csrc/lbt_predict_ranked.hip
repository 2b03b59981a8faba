// PredictTask for large inputs: the rows' values are replaced by their ranks among the ensemble's thresholds once,
// and the walk compares ranks.
//
// Semantics: rapidsai/legate-boost src/models/tree/predict.cu:26-84, bit for bit: x <= t holds exactly when
// #{thresholds of the feature < x} <= #{thresholds of the feature < t} (both over the whole ensemble, equal ones
// counted as often as they occur), and a row's leaf values are added in tree order.
//
// What bounds a walk is how often it goes to the LDS: every step reads a node and a value. predict_tile_kernel reads 8-byte nodes
// and 4- or 8-byte values of a row tile in row order, 16.7 cycles of a CU per wave and step (20,000,000 x 64, 1000 trees of
// depth 8: 67.9 ms). With ranks of 16 bits a node is one word (rank, feature), a value is two bytes, four times as
// many rows share a copied node, a lane keeps one row (its value of any feature lies in the lane's own bank) and
// adds its own leaf values, and the tree is a complete heap, so that no child index is stored: 7 cycles, 29.6 ms, and
// 2.8 ms for the ranks. The LDS is then busy for 74 % of the time (8 % conflicts), the vector units (4.4 instructions a step)
// for 62 %, and the L1 looks up 0.66 lines a cycle (profiles/predict_ranked_cfg5_20Mx64_1000trees.txt); reads in two
// staggered halves (30.7 ms) and rank loads into the upper half of a register (34.5) were no faster.
#include "lbt_internal.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "lbt_trees.h"

namespace lbt {
namespace {

constexpr int kThreads       = 256;
constexpr int kWalkThreads   = 1024;
constexpr int kWalkWaves     = kWalkThreads / 64;
constexpr int kPackTrees     = 64;    // trees packed per launch (descriptors passed by value)
constexpr int kMaxPerFeature = 65533; // thresholds of a feature: ranks 1 .. count + 1 below the rank of a NaN
constexpr uint32_t kNanRank  = 0xffffu;
constexpr int kRankBlocks    = 16;    // workgroups that share the ranking of a feature's thresholds
constexpr int kRankTile      = 2048;  // thresholds in the LDS at a time
constexpr size_t kLds        = 160 * 1024 - 2048;
constexpr int kGroupMax      = 8;     // features a lane of the rank pass takes at once

struct PackRefs {
  const double* leaf[kPackTrees];
  const int32_t* feature[kPackTrees];
  const double* split[kPackTrees];
  int32_t n_nodes[kPackTrees];
};

struct RankState {
  int depth, F, K, n_trees;  // n_trees: padded to whole chunks
  int32_t* count;       // [F] thresholds of a feature; [F] not 0 where a node on the feature has NaN as its threshold
  int32_t* offset;      // [F + 1]
  int32_t* overflow;    // one word: a feature has more thresholds than ranks
  uint32_t* slot;       // [n_trees << depth] place among the thresholds of the node's feature, or a marker
  uint32_t* nodes;      // [n_trees << depth] first the feature, then rank << 16 | feature; heap order, root at 1
  double* leaves;       // [n_trees << depth][K]
  uint32_t* owner;      // [thresholds] node of a threshold, by feature
};
constexpr uint32_t kNoThreshold = 0xffffffffu;

__global__ void zero_counts_kernel(int32_t* count, int n)
{
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < n) count[i] = 0;
}

// One thread per heap slot of a tree of `depth` complete levels: slot i is inner node i (1 is the root) and leaf i of the
// bottom. What lies below a node that ends the walk is never decisive: every bottom leaf below it has its value.
// A workgroup takes kTogether trees and counts their thresholds in the LDS (when kLocal: the counters fit), so that
// a feature's counter in memory is added to once per workgroup and not once per node: adds to one address take turns
// of about 0.1 us (64 trees of depth 8 on 64 features: 29 us a launch with an add per node and a chain of loads, 14 now).
constexpr int kPackTogether  = 4;
constexpr int kLeafLoads     = 8;
constexpr int kLocalCounters = 8192;
template <typename T, bool kLocal, int kTogether>
__global__ void __launch_bounds__(kThreads) rank_pack_kernel(PackRefs refs, int first, int here, int all, RankState st, T* raw)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  int32_t* s_count = reinterpret_cast<int32_t*>(smem_raw);
  const int i      = blockIdx.x * kThreads + threadIdx.x;
  const int size   = 1 << st.depth;
  if constexpr (kLocal) {
    for (int f = threadIdx.x; f < st.F; f += kThreads) s_count[f] = 0;
    __syncthreads();
  }
  int slot[kTogether], node_feature[kTogether];
#pragma unroll
  for (int u = 0; u < kTogether; u++) {
    const int t     = blockIdx.y * kTogether + u;
    slot[u]         = -1;
    node_feature[u] = 0;
    if (i >= size || t >= all) continue;
    const int64_t at = (static_cast<int64_t>(first + t) << st.depth) + i;
    if (t >= here) continue;  // padding to whole chunks: a tree whose values nothing adds
    const int32_t* feature = refs.feature[t];
    const int n            = refs.n_nodes[t];
    auto ends = [&](int node) {
      // a node whose children would lie past the arrays, or whose feature does not exist, ends the walk
      const int ft = feature[min(node, n - 1)];
      return (node >= n) | (ft < 0) | (ft >= st.F) | (2 * static_cast<int64_t>(node) + 2 >= n);
    };
    // which nodes above bottom leaf i, and above and at inner node i, end the walk; none of the loads waits for another
    uint32_t ends_leaf = 0, ends_node = 0;
    const int level = i > 0 ? 31 - __clz(i) : -1;
#pragma unroll 4
    for (int l = 0; l < st.depth; l++) {
      ends_leaf |= static_cast<uint32_t>(ends(((size + i) >> (st.depth - l)) - 1)) << l;
      if (l <= level) ends_node |= static_cast<uint32_t>(ends((i >> (level - l)) - 1));
    }
    if (i > 0 && ends_node == 0) {
      const int ft   = feature[i - 1];
      const double d = refs.split[t][i - 1];
      T thr;
      if constexpr (sizeof(T) == 4)
        thr = round_down_to_float(d);
      else
        thr = d;
      node_feature[u] = ft;
      if (thr == thr) {
        slot[u] = kLocal ? atomicAdd(&s_count[ft], 1) : atomicAdd(&st.count[ft], 1);
        raw[at] = thr;
      } else {
        // a comparison with NaN is never true: rank 0, below every value's; the feature then needs ranks, whatever they are
        st.count[st.F + ft] = 1;
      }
    }
    const int stop = ends_leaf != 0 ? __ffs(ends_leaf) - 1 : st.depth;
    const int a    = (size + i) >> (st.depth - stop);
    // (loads of several outputs under way together: hipcc has every load wait behind the store before it, and with eight outputs
    // 50 trees took 24 us that way, 21.5 this way; of one output there is one, not eight of the same)
    const double* from = refs.leaf[t] + static_cast<int64_t>(a - 1) * st.K;
    double* to         = st.leaves + at * st.K;
    if (st.K == 1) {
      *to = *from;
      continue;
    }
    for (int k0 = 0; k0 < st.K; k0 += kLeafLoads) {
      double v[kLeafLoads];
#pragma unroll
      for (int k = 0; k < kLeafLoads; k++) v[k] = from[min(k0 + k, st.K - 1)];
#pragma unroll
      for (int k = 0; k < kLeafLoads; k++)
        if (k0 + k < st.K) to[k0 + k] = v[k];
    }
  }
  if constexpr (kLocal) {
    __syncthreads();
    for (int f = threadIdx.x; f < st.F; f += kThreads) {
      const int n = s_count[f];
      s_count[f]  = n > 0 ? atomicAdd(&st.count[f], n) : 0;
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < kTogether; u++) {
    const int t = blockIdx.y * kTogether + u;
    if (i >= size || t >= all) continue;
    const int64_t at = (static_cast<int64_t>(first + t) << st.depth) + i;
    const int base   = kLocal && slot[u] >= 0 ? s_count[node_feature[u]] : 0;
    st.slot[at]      = slot[u] >= 0 ? static_cast<uint32_t>(base + slot[u]) : kNoThreshold;
    st.nodes[at]     = static_cast<uint32_t>(node_feature[u]);
  }
}

// exclusive sums of the features' counts; one workgroup
__global__ void __launch_bounds__(1024) rank_offsets_kernel(RankState st)
{
  __shared__ int32_t s_sum[1024];
  __shared__ int s_over;
  const int tid = threadIdx.x, per = (st.F + 1023) / 1024;
  if (tid == 0) s_over = 0;
  __syncthreads();
  int sum = 0;
  for (int i = 0; i < per; i++) {
    const int f = tid * per + i;
    if (f < st.F) {
      sum += st.count[f];
      if (st.count[f] > kMaxPerFeature) s_over = 1;
    }
  }
  s_sum[tid] = sum;
  __syncthreads();
  for (int d = 1; d < 1024; d *= 2) {
    const int32_t v = tid >= d ? s_sum[tid - d] : 0;
    __syncthreads();
    s_sum[tid] += v;
    __syncthreads();
  }
  int at = tid > 0 ? s_sum[tid - 1] : 0;
  for (int i = 0; i < per; i++) {
    const int f = tid * per + i;
    if (f < st.F) {
      st.offset[f] = at;
      at += st.count[f];
    }
  }
  if (tid == 1023) st.offset[st.F] = s_sum[1023];
  if (tid == 0) *st.overflow = s_over;
}

template <typename T>
__global__ void __launch_bounds__(kThreads) rank_scatter_kernel(RankState st, const T* raw, T* grouped)
{
  const int64_t i = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  if (i >= static_cast<int64_t>(st.n_trees) << st.depth) return;
  const uint32_t slot = st.slot[i];
  if (slot == kNoThreshold) return;
  const int at  = st.offset[st.nodes[i]] + static_cast<int>(slot);
  grouped[at]   = raw[i];
  st.owner[at]  = static_cast<uint32_t>(i);
}

// number of values of tab[0 .. m) below x
template <typename T>
__device__ inline int lower_bound(const T* tab, int m, T x)
{
  if (m == 0) return 0;
  const int top = 1 << (31 - __clz(m));
  int at        = tab[top - 1] < x ? m - top + 1 : 0;
  for (int step = top >> 1; step > 0; step >>= 1) at += tab[at + step - 1] < x ? step : 0;
  return at;
}

// The rank of a threshold is the number of smaller ones of its feature. A feature's thresholds are sorted in the LDS of one
// workgroup (bitonic; owners move along); where they are too many for it the feature's workgroups count instead,
// comparing each with all (1000 trees of depth 8 on 64 features, 4000 thresholds a feature: 213 us by counting, 97 sorted).
constexpr int kSortThreads = 1024;
template <typename T>
constexpr int kSortMost = sizeof(T) == 4 ? 16384 : 8192;
template <typename T>
__global__ void __launch_bounds__(kSortThreads) rank_thresholds_kernel(RankState st, int sort_most, const T* grouped, T* sorted)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  if (*st.overflow != 0) return;
  const int tid = threadIdx.x, f = blockIdx.x, first = st.offset[f], m = st.offset[f + 1] - first;
  T* s_val = reinterpret_cast<T*>(smem_raw);
  if (m <= sort_most) {
    if (blockIdx.y != 0 || m == 0) return;
    uint32_t* s_owner = reinterpret_cast<uint32_t*>(s_val + sort_most);
    int size = 2;
    while (size < m) size *= 2;
    for (int i = tid; i < size; i += kSortThreads) {
      s_val[i]   = i < m ? grouped[first + i] : static_cast<T>(__builtin_huge_val());
      s_owner[i] = i < m ? st.owner[first + i] : kNoThreshold;
    }
    for (int width = 2; width <= size; width *= 2)
      for (int d = width / 2; d > 0; d /= 2) {
        __syncthreads();
        for (int p = tid; p < size / 2; p += kSortThreads) {
          const int i = 2 * p - (p & (d - 1)), j = i + d;
          const T a = s_val[i], b = s_val[j];
          const uint32_t oa = s_owner[i], ob = s_owner[j];
          // the padding (infinity without an owner) stays behind thresholds that are infinite
          const bool above = a > b || (a == b && oa > ob);
          if (above == ((i & width) == 0)) {
            s_val[i]   = b;
            s_val[j]   = a;
            s_owner[i] = ob;
            s_owner[j] = oa;
          }
        }
      }
    __syncthreads();
    for (int i = tid; i < m; i += kSortThreads) {
      const T v                  = s_val[i];
      sorted[first + i]          = v;
      const int less             = lower_bound(s_val, m, v);
      st.nodes[s_owner[i]]       = (static_cast<uint32_t>(less + 1) << 16) | static_cast<uint32_t>(f);
    }
    return;
  }
  for (int e0 = blockIdx.y * kSortThreads; e0 < m; e0 += gridDim.y * kSortThreads) {
    const int e = e0 + tid;
    const T v   = e < m ? grouped[first + e] : T(0);
    int less = 0, same = 0;
    for (int b = 0; b < m; b += kRankTile) {
      const int n = min(kRankTile, m - b);
      __syncthreads();
      for (int i = tid; i < n; i += kSortThreads) s_val[i] = grouped[first + b + i];
      __syncthreads();
#pragma unroll 8
      for (int i = 0; i < n; i++) {
        const T o = s_val[i];
        less += o < v ? 1 : 0;
        same += o == v && b + i < e ? 1 : 0;
      }
    }
    if (e < m) {
      sorted[first + less + same] = v;
      st.nodes[st.owner[first + e]] = (static_cast<uint32_t>(less + 1) << 16) | static_cast<uint32_t>(f);
    }
  }
}

// ---- the rows' ranks

struct RankRows {
  int64_t n_rows;   // of the chunk
  int F, n_groups, tile_shift, cells;
  int64_t rows_per_split;  // a multiple of the threads
  int lds_bytes;
  int wide;         // X rows can be read 16 bytes at a time
};

// what a wave has written to the LDS is read by its other lanes
__device__ __forceinline__ void wave_lds_fence()
{
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The first guess at the place of x among the thresholds: cells of one width between the smallest and the largest, each with
// the number of thresholds in the cells before it. The cell of a value never falls as the value rises (each
// operation rounds monotonically; NaN, from 0 * infinity or infinities, goes to cell 0 for thresholds and values
// alike), so thresholds of lower cells are below x and those of higher ones above it, however they are spread.
template <typename T>
__device__ __forceinline__ int cell_of(T x, T lo, T scale, int cells)
{
  const T c = (x - lo) * scale;
  return static_cast<int>(fmin(fmax(c, T(0)), static_cast<T>(cells - 1)));
}

// Place of a row among the tile's ranks of a feature. The LDS serves the lanes 0 .. 31 of a wave at once, 4 bytes a bank:
// rows r and r + 32 of a wave share a word, so that those lanes read 32 banks whatever features they ask for.
__device__ __forceinline__ int row_place(int row) { return (row & ~63) + 2 * (row & 31) + ((row >> 5) & 1); }

// Stores a wave's ranks of its 64 rows (a block of 64 of a tile) for kN neighbouring features, of which `here` exist: the lanes of two features exchange
// halves, so that a lane holds the two rows of a word and a store is two whole cache lines. `to`: the block's word 0 of the first
// feature. All lanes take part; what rows past the last one get is never read. (Where the search is what bounds a pass it gained
// nothing: 20,000,000 x 64, eight features a lane, 2.56 ms with stores of two bytes, 2.63 with these.)
template <int kN>
__device__ __forceinline__ void store_ranks(const uint32_t (&code)[kN], int here, int tile_shift, char* to)
{
  const int lane = threadIdx.x & 63;
  static_assert(kN % 2 == 0, "features in pairs");
#pragma unroll
  for (int j = 0; j < kN; j += 2) {
    // of the second feature the lower lanes, of the first one the upper lanes
    const auto swapped = __builtin_amdgcn_permlane32_swap(code[j], code[j + 1], false, false);
    const int f        = j + (lane >> 5);
    if (f < here)
      *reinterpret_cast<uint32_t*>(to + ((static_cast<uint32_t>(2 * f) << tile_shift) + 4u * (static_cast<uint32_t>(lane) & 31u))) =
        swapped[0] | swapped[1] << 16;
  }
}

// What a workgroup's searches begin with: for each of its kAll features the cells' first places, how many probes tell the places of a
// cell from one another, and the cell function. s_place, s_count: where its thresholds begin and how many there are. A wave per feature.
template <typename T, int kAll>
__device__ __forceinline__ void rank_cells(int cells, const T* s_tab, uint16_t* s_start, const int (&s_place)[kAll], const int (&s_count)[kAll],
                                           int (&s_most)[kAll], T (&s_lo)[kAll], T (&s_scale)[kAll])
{
  const int tid = threadIdx.x;
  for (int i = tid >> 6; i < kAll; i += kWalkWaves) {
    const int m = s_count[i], lane = tid & 63;
    if (m == 0) {
      if (lane == 0) s_lo[i] = s_scale[i] = T(0);
      continue;
    }
    const T* tab    = s_tab + s_place[i];
    uint16_t* start = s_start + i * cells;
    T lo            = tab[0];
    T scale         = static_cast<T>(cells) / (tab[m - 1] - lo);
    // the first threshold of a cell counts those before it, for that cell and the empty ones below it
    int most = 0;
    for (int e = lane; e < m; e += 64) {
      const int c = cell_of(tab[e], lo, scale, cells);
      const int p = e == 0 ? -1 : cell_of(tab[e - 1], lo, scale, cells);
      for (int b = p + 1; b <= c; b++) start[b] = static_cast<uint16_t>(e);
      if (e == m - 1)
        for (int b = c + 1; b < cells; b++) start[b] = static_cast<uint16_t>(m);
    }
    wave_lds_fence();
    for (int c = lane; c < cells; c += 64) most = max(most, (c + 1 < cells ? start[c + 1] : m) - start[c]);
    for (int d = 32; d > 0; d /= 2) most = max(most, __shfl_xor(most, d, 64));
    int probes = 32 - __clz(most);  // they tell 2^probes places from one another
    wave_lds_fence();
    if ((1 << probes) - 1 > m) {
      // nearly all in one cell: two cells instead, below and above the threshold that a plain search asks first
      probes = 31 - __clz(m);
      lo     = tab[(1 << probes) - 1];
      scale  = static_cast<T>(__builtin_huge_val());
      for (int c = lane; c < cells; c += 64) start[c] = c == cells - 1 ? 0xffff : 0;
    }
    // a search may begin earlier (the thresholds before its cell are below x), and must where it would probe past the end
    const int last = m + 1 - (1 << probes);
    for (int c = lane; c < cells; c += 64) start[c] = static_cast<uint16_t>(min(static_cast<int>(start[c]), last));
    if (lane == 0) {
      s_most[i]  = probes;
      s_lo[i]    = lo;
      s_scale[i] = scale;
    }
  }
}

// A workgroup has the thresholds of kGroup neighbouring features in its LDS and a lane takes its row's values of those. The
// workgroups of one row range are neighbours on one XCD, so that they find a line that several of them ask for in its L2.
// ranks: [tile][feature][place of the row]
// What bounds it are the LDS and vector instructions, a read and four instructions per probe of a search and feature. With cells to start
// from a feature of 4000 evenly spread thresholds takes 4 or 5 probes instead of 12 (20,000,000 x 64: 6.1 ms without cells, 2.8 with, 2.56
// since features with fewer probes take no part in the others').
template <typename T, int kAll>
__global__ void __launch_bounds__(kWalkThreads, 4)
  rank_rows_kernel(const T* __restrict__ X, RankRows a, RankState st, const T* __restrict__ sorted,
                   uint16_t* __restrict__ ranks)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ int s_most[kAll], s_place[kAll], s_count[kAll];
  __shared__ T s_lo[kAll], s_scale[kAll];
  if (*st.overflow != 0) return;
  const int tid = threadIdx.x, local = blockIdx.x / 8, g = local % a.n_groups;
  const int64_t split = blockIdx.x % 8 + 8 * static_cast<int64_t>(local / a.n_groups);
  const int f0 = g * kAll, nf = min(kAll, a.F - f0);
  const int first = st.offset[f0], words = st.offset[f0 + nf] - first;
  if (words == 0) {
    bool asked = false;
    for (int i = 0; i < nf; i++) asked |= st.count[a.F + f0 + i] != 0;
    if (!asked) return;  // no tree asks for these features
  }
  T* const s_tab    = reinterpret_cast<T*>(smem_raw);
  uint16_t* s_start = reinterpret_cast<uint16_t*>(smem_raw + a.lds_bytes - 2 * kAll * a.cells);  // [kAll][cells]
  const bool held   = (words + 1) * static_cast<int>(sizeof(T)) + 2 * kAll * a.cells <= a.lds_bytes;
  if (tid < kAll) {
    const int at = st.offset[f0 + min(tid, nf)];
    s_most[tid]  = 0;
    s_place[tid] = at - first;
    s_count[tid] = tid < nf ? st.offset[f0 + tid + 1] - at : 0;
  }
  if (held) {
    for (int e = tid; e < words; e += kWalkThreads) s_tab[e] = sorted[first + e];
    if (tid == 0) s_tab[words] = T(0);  // read, not used, by features without thresholds
    for (int c = tid; c < kAll * a.cells; c += kWalkThreads) s_start[c] = 0;
  }
  __syncthreads();
  if (held) rank_cells<T, kAll>(a.cells, s_tab, s_start, s_place, s_count, s_most, s_lo, s_scale);
  __syncthreads();
  const int64_t end = min<int64_t>(a.n_rows, (split + 1) * a.rows_per_split);
  typedef T Vec __attribute__((ext_vector_type(16 / sizeof(T))));
  constexpr int kPer = 16 / sizeof(T);
  auto load = [&](int64_t row, T (&x)[kAll]) {
    const T* src = X + row * a.F + f0;
    if (a.wide) {
      // rows of whole 16-byte words: a word lies inside the features or past them
#pragma unroll
      for (int i = 0; i < kAll / kPer; i++) {
        const Vec v = reinterpret_cast<const Vec*>(src)[i * kPer < nf ? i : 0];
#pragma unroll
        for (int j = 0; j < kPer; j++) x[i * kPer + j] = v[j];
      }
    } else {
#pragma unroll
      for (int i = 0; i < kAll; i++) x[i] = src[i < nf ? i : 0];
    }
  };
  int place[kAll], probes[kAll], most_probes = 0;
  T lo[kAll], scale[kAll];
#pragma unroll
  for (int i = 0; i < kAll; i++) {
    place[i]    = __builtin_amdgcn_readfirstlane(s_place[i]);
    probes[i]   = __builtin_amdgcn_readfirstlane(s_most[i]);
    lo[i]       = s_lo[i];
    scale[i]    = s_scale[i];
    most_probes = max(most_probes, probes[i]);
  }
  int64_t row = split * a.rows_per_split + tid;
  T x[kAll], next[kAll];
  if (row < end) load(row, next);
  for (; row < end; row += kWalkThreads) {
#pragma unroll
    for (int i = 0; i < kAll; i++) x[i] = next[i];
    if (row + kWalkThreads < end) load(row + kWalkThreads, next);
    // tile rows are a power of two; a tile's ranks lie within 32 bits of bytes
    const int64_t tile = row >> a.tile_shift;
    char* base         = reinterpret_cast<char*>(ranks + (tile * a.F + f0) * (int64_t(1) << a.tile_shift));
    const uint32_t at0 = 2 * row_place(static_cast<int>(row) & ((1 << a.tile_shift) - 1));
    int at[kAll];
    if (held) {
#pragma unroll
      for (int i = 0; i < kAll; i++) at[i] = s_start[i * a.cells + cell_of(x[i], lo[i], scale[i], a.cells)];
      for (int p = most_probes - 1; p >= 0; p--) {
#pragma unroll
        for (int i = 0; i < kAll; i++) {
          if (p >= probes[i]) continue;  // (the same for the whole wave)
          const T v = s_tab[place[i] + ((1 << p) - 1) + at[i]];
          at[i] += v < x[i] ? 1 << p : 0;
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < kAll; i++) at[i] = lower_bound(sorted + first + s_place[i], s_count[i], x[i]);
    }
#pragma unroll
    for (int i = 0; i < kAll; i++) {
      const uint32_t code = x[i] == x[i] ? static_cast<uint32_t>(at[i]) + 1 : kNanRank;
      if (i < nf)
        *reinterpret_cast<uint16_t*>(base + (at0 + (static_cast<uint32_t>(2 * i) << a.tile_shift))) = static_cast<uint16_t>(code);
    }
  }
}

// The same for the features of one 128-byte line of a row, where their tables leave two such workgroups to a CU. Eight lanes take a row's
// line, 16 bytes each: a wave's load so touches eight whole lines (a row a lane touched 64, once for each of its eight loads of 16
// bytes: without any search 500,003 x 200 took 186 of 202 us that way). The values are turned in the LDS, and then a lane has a row and a
// wave two, four or eight features, whose search it keeps in scalar registers; the rows of one feature share many of its LDS reads.
// What bounds it is the memory: 500,003 x 200 (0.6 GB) 156 us. A line with more thresholds than there is room for beside the rows has fewer cells,
// a probe more for each half of them, before it falls to a search in memory, every probe a load: 50 trees of depth 8 on 2,000,000 x 200, a share of 0.6 of
// the thresholds on one line of floats 1204 us a call (2180 searched in memory, 1104 evenly), of 0.33 on one line of doubles 1525 (3377, 1456).
constexpr int kFewCells = 64;  // cells of a feature at least
template <typename T>
constexpr int kLineFeatures = 128 / sizeof(T);
// kRows: rows of a turn
template <typename T, int kRows>
constexpr int kLinePitch = kRows + (sizeof(T) == 4 ? 2 : 4);  // the eight lanes of a row, eight rows: 64 banks
template <typename T, int kRows>
constexpr int kLineStage = kLineFeatures<T> * kLinePitch<T, kRows> * static_cast<int>(sizeof(T));
inline size_t line_stage(size_t value_size, int rows)
{
  return value_size == 4 ? kLineStage<float, 256> : (rows == 256 ? kLineStage<double, 256> : kLineStage<double, 128>);
}
template <typename T, int kRows>
__global__ void __launch_bounds__(kWalkThreads, 8)
  rank_lines_kernel(const T* __restrict__ X, RankRows a, RankState st, const T* __restrict__ sorted, uint16_t* __restrict__ ranks)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int kAll = kLineFeatures<T>, kPer = 16 / sizeof(T), kPitch = kLinePitch<T, kRows>;
  constexpr int kLoads = kRows * 8 / kWalkThreads, kShares = kWalkWaves / (kRows / 64);  // of a thread; waves that share a row's features
  __shared__ int s_most[kAll], s_place[kAll], s_count[kAll];
  __shared__ T s_lo[kAll], s_scale[kAll];
  if (*st.overflow != 0) return;
  const int tid = threadIdx.x, local = blockIdx.x / 8, g = local % a.n_groups;
  const int64_t split = blockIdx.x % 8 + 8 * static_cast<int64_t>(local / a.n_groups);
  const int f0 = g * kAll, nf = min(kAll, a.F - f0);
  const int first = st.offset[f0], words = st.offset[f0 + nf] - first;
  if (words == 0) {
    bool asked = false;
    for (int i = 0; i < nf; i++) asked |= st.count[a.F + f0 + i] != 0;
    if (!asked) return;  // no tree asks for these features
  }
  // a lane's piece of its rows
  const int q = tid & 7, r = tid >> 3, fq = f0 + kPer * q;  // rows r + 128 u
  const int64_t begin = split * a.rows_per_split, end = min<int64_t>(a.n_rows, begin + a.rows_per_split);
  typedef T Vec __attribute__((ext_vector_type(kPer)));
  auto load = [&](int64_t row, T (&x)[kPer]) {
    const T* src = X + min(row, end - 1) * a.F;
    if (a.wide) {
      // rows of whole 16-byte words: a word lies inside the features or past them
      const Vec v = *reinterpret_cast<const Vec*>(src + (fq < a.F ? fq : f0));
#pragma unroll
      for (int j = 0; j < kPer; j++) x[j] = v[j];
    } else {
#pragma unroll
      for (int j = 0; j < kPer; j++) x[j] = src[min(fq + j, a.F - 1)];
    }
  };
  T ahead[kLoads][kPer];
  auto load_turn = [&](int64_t row0) {
#pragma unroll
    for (int u = 0; u < kLoads; u++) load(row0 + r + u * (kWalkThreads / 8), ahead[u]);
  };
  if (begin < end) load_turn(begin);
  // Tables beside the turned rows, with fewer cells if need be, or else in memory.
  const int table = (words + 1) * static_cast<int>(sizeof(T));
  int cells       = a.cells;
  while (cells > kFewCells && table + 2 * kAll * cells > a.lds_bytes) cells /= 2;
  const bool held   = table + 2 * kAll * cells <= a.lds_bytes;
  T* const s_x      = reinterpret_cast<T*>(smem_raw);  // [kAll][kPitch]
  T* const s_tab    = reinterpret_cast<T*>(smem_raw + kLineStage<T, kRows>);
  uint16_t* s_start = reinterpret_cast<uint16_t*>(smem_raw + kLineStage<T, kRows> + a.lds_bytes - 2 * kAll * cells);  // [kAll][cells]
  if (tid < kAll) {
    const int at = st.offset[f0 + min(tid, nf)];
    s_most[tid]  = 0;
    s_place[tid] = at - first;
    s_count[tid] = tid < nf ? st.offset[f0 + tid + 1] - at : 0;
  }
  if (held) {
    for (int e = tid; e < words; e += kWalkThreads) s_tab[e] = sorted[first + e];
    if (tid == 0) s_tab[words] = T(0);  // read, not used, by features without thresholds
    for (int c = tid; c < kAll * cells; c += kWalkThreads) s_start[c] = 0;
  }
  __syncthreads();
  if (held) rank_cells<T, kAll>(cells, s_tab, s_start, s_place, s_count, s_most, s_lo, s_scale);
  __syncthreads();
  // a wave's features of 64 rows
  constexpr int kOwn = kAll / kShares;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), own = wave % kShares * kOwn, row_of = wave / kShares * 64 + (tid & 63);
  int place[kOwn], probes[kOwn], most_probes = 0;
  T lo[kOwn], scale[kOwn];
  auto uniform = [](T v) {
    uint32_t w[sizeof(T) / 4];
    __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
    for (uint32_t& u : w) u = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(u)));
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
  };
#pragma unroll
  for (int j = 0; j < kOwn; j++) {
    place[j]    = __builtin_amdgcn_readfirstlane(s_place[own + j]);
    probes[j]   = __builtin_amdgcn_readfirstlane(s_most[own + j]);
    lo[j]       = uniform(s_lo[own + j]);
    scale[j]    = uniform(s_scale[own + j]);
    most_probes = max(most_probes, probes[j]);
  }
  const uint16_t* const start = s_start + own * cells;
  for (int64_t row0 = begin; row0 < end; row0 += kRows) {
#pragma unroll
    for (int u = 0; u < kLoads; u++)
#pragma unroll
      for (int j = 0; j < kPer; j++) s_x[(kPer * q + j) * kPitch + r + u * (kWalkThreads / 8)] = ahead[u][j];
    if (row0 + kRows < end) load_turn(row0 + kRows);
    __syncthreads();
    T x[kOwn];
    int at[kOwn];
#pragma unroll
    for (int j = 0; j < kOwn; j++) x[j] = s_x[(own + j) * kPitch + row_of];
    if (held) {
#pragma unroll
      for (int j = 0; j < kOwn; j++) at[j] = start[j * cells + cell_of(x[j], lo[j], scale[j], cells)];
      for (int p = most_probes - 1; p >= 0; p--) {
#pragma unroll
        for (int j = 0; j < kOwn; j++) {
          if (p >= probes[j]) continue;  // (the same for the whole wave)
          const T v = s_tab[place[j] + ((1 << p) - 1) + at[j]];
          at[j] += v < x[j] ? 1 << p : 0;
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < kOwn; j++) at[j] = lower_bound(sorted + first + place[j], s_count[own + j], x[j]);
    }
    const int64_t block = row0 + wave / kShares * 64;  // (a split ends with a block, or with the last row)
    if (block < end) {
      uint32_t code[kOwn];
#pragma unroll
      for (int j = 0; j < kOwn; j++) code[j] = x[j] == x[j] ? static_cast<uint32_t>(at[j]) + 1 : kNanRank;
      // tile rows are a power of two, 64 or more; a tile's ranks lie within 32 bits of bytes
      const int64_t tile = block >> a.tile_shift;
      char* const base   = reinterpret_cast<char*>(ranks + (tile * a.F + f0 + own) * (int64_t(1) << a.tile_shift));
      store_ranks(code, nf - own, a.tile_shift, base + 2 * (static_cast<int>(block) & ((1 << a.tile_shift) - 1)));
    }
    __syncthreads();
  }
}

// ---- the walk

struct WalkArgs {
  int64_t n_rows;
  int F, K, depth, n_trees, tile_rows;
  int chunk;       // trees in the LDS at a time: a multiple of (waves per row) * kJ
  int node_off, index_off, acc_off;  // where the LDS has the nodes and, for two chunks, the leaf numbers or values; the sums
};

typedef unsigned int Word16 __attribute__((ext_vector_type(4)));
constexpr int kLeavesInLds = 2;
constexpr int kWalkCopy = 4;  // 16-byte words a thread moves per chunk

// low half of a * b + c in one instruction (there is no builtin for it)
__device__ __forceinline__ uint32_t mad_u32_u16(uint32_t a, uint32_t b, uint32_t c)
{
  uint32_t r;
  asm("v_mad_u32_u16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
  return r;
}

// LDS by its 32-bit address: the walk's address arithmetic then is what is written below and no more
template <typename T>
using LdsPtr = const __attribute__((address_space(3))) T*;
template <typename T>
__device__ __forceinline__ LdsPtr<T> lds_at(uint32_t address)
{
  return reinterpret_cast<LdsPtr<T>>(static_cast<uintptr_t>(address));
}
__device__ __forceinline__ uint32_t lds_address(unsigned char* p)
{
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)p));
}

// Walks kJ trees of the LDS at once. pos: heap index, from the root 1 to the bottom 2^depth + leaf. Four vector
// instructions per step and tree: node address, value address, difference of the ranks (negative: to the right),
// and its sign shifted into the heap index.
// nodes, lane_x: LDS addresses of the first tree and of the lane's row.
template <int kJ>
__device__ __forceinline__ void walk_trees(uint32_t (&pos)[kJ], uint32_t nodes, int depth, uint32_t lane_x, uint32_t stride)
{
#pragma unroll
  for (int j = 0; j < kJ; j++) pos[j] = 1;
  for (int s = 0; s < depth; s++) {
    uint32_t nd[kJ], x[kJ];
#pragma unroll
    for (int j = 0; j < kJ; j++) nd[j] = *lds_at<uint32_t>(4 * pos[j] + (nodes + (j << (depth + 2))));
    __builtin_amdgcn_sched_barrier(0);  // all trees' nodes are asked for before the first is waited for
#pragma unroll
    for (int j = 0; j < kJ; j++) x[j] = *lds_at<uint16_t>(mad_u32_u16(nd[j], stride, lane_x));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < kJ; j++) pos[j] = __builtin_amdgcn_alignbit(pos[j], (nd[j] >> 16) - x[j], 31);
  }
}

// Who adds the leaf values of a row, in tree order:
//   kOwn       one output, a row per lane: the lane that walks all its trees
//   kInTurn    one output, several waves per row: leaf numbers pass through the LDS and one of the waves adds a chunk's values
//              while the next chunk is walked, another wave every chunk; the sums lie in the LDS
//   kShared    several outputs: (row, output) sums are shared out among the lanes, kItems each, output fastest
enum class Adds { kOwn, kInTurn, kShared };

template <Adds kAdds, int kItems, int kJ>
__global__ void __launch_bounds__(kWalkThreads)
  walk_ranked_kernel(const uint16_t* __restrict__ ranks, WalkArgs a, RankState st, double* __restrict__ out)
{
  constexpr bool kOwn = kAdds == Adds::kOwn;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  if (*st.overflow != 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int R = a.tile_rows, row_waves = R / 64, tree_waves = kWalkWaves / row_waves;
  const int rw = kOwn ? wave : wave % row_waves, tw = kOwn ? 0 : wave / row_waves;
  const int64_t row0  = blockIdx.x * static_cast<int64_t>(R);
  const int rows_here = static_cast<int>(min<int64_t>(R, a.n_rows - row0));
  const int my_row    = rw * 64 + lane;
  const int n16       = (a.chunk << a.depth) / 4;
  Word16 pf[kWalkCopy], pf_leaf;
  // kOwn: the leaf values of the first kLdsLeaves of kJ trees come from the LDS, those of the others from the L1, whose
  // 46 line look-ups per gather would else be the longest of the three (vector instructions, LDS, L1)
  constexpr int kLdsLeaves = kOwn && kJ == 8 ? kLeavesInLds : 0;
  const int n16_leaf       = kLdsLeaves << a.depth >> 1;
  auto fetch = [&](int first) {
    if (kLdsLeaves > 0 && tid < n16_leaf)
      pf_leaf = reinterpret_cast<const Word16*>(st.leaves + (static_cast<int64_t>(first) << a.depth))[tid];
    const Word16* src = reinterpret_cast<const Word16*>(st.nodes + (static_cast<int64_t>(first) << a.depth));
#pragma unroll
    for (int c = 0; c < kWalkCopy; c++)
      if (tid + c * kWalkThreads < n16) pf[c] = src[tid + c * kWalkThreads];
  };
  auto store = [&](int buf) {
    if (kLdsLeaves > 0 && tid < n16_leaf) (reinterpret_cast<Word16*>(smem_raw + a.index_off) + buf * n16_leaf)[tid] = pf_leaf;
    Word16* dst = reinterpret_cast<Word16*>(smem_raw + a.node_off) + buf * n16;
#pragma unroll
    for (int c = 0; c < kWalkCopy; c++)
      if (tid + c * kWalkThreads < n16) dst[tid + c * kWalkThreads] = pf[c];
  };
  fetch(0);
  {
    const Word16* src = reinterpret_cast<const Word16*>(ranks + static_cast<int64_t>(blockIdx.x) * R * a.F);
    Word16* dst       = reinterpret_cast<Word16*>(smem_raw);
    const int n       = R * a.F / 8;
#pragma unroll 4
    for (int i = tid; i < n; i += kWalkThreads) dst[i] = src[i];
  }
  store(0);
  uint16_t* const s_index = reinterpret_cast<uint16_t*>(smem_raw + a.index_off);  // [2][chunk][R]
  double* const s_acc     = reinterpret_cast<double*>(smem_raw + a.acc_off);      // kInTurn: [R]
  if (kAdds == Adds::kInTurn && tw == 0) s_acc[my_row] = 0.0;
  __syncthreads();
  const uint32_t lds_base = lds_address(smem_raw);
  const uint32_t lane_x   = lds_base + 2 * row_place(my_row);  // the ranks lie at the start of the LDS
  const uint32_t stride   = 2 * R;
  const int per_wave      = a.chunk / tree_waves;  // trees of a chunk this wave walks

  // kShared: this lane's sums
  const int per_items = R * a.K / kWalkWaves;
  double acc[kItems];
  int item_row[kItems], item_out[kItems];
#pragma unroll
  for (int i = 0; i < kItems; i++) {
    const int v = wave * per_items + min(lane + 64 * i, per_items - 1);
    acc[i]      = 0.0;
    item_row[i] = kAdds == Adds::kShared ? v / a.K : my_row;
    item_out[i] = kAdds == Adds::kShared ? v - item_row[i] * a.K : 0;
  }
  // values of kAhead trees of a chunk from tree c on
  constexpr int kAhead = kAdds == Adds::kInTurn ? 16 : 8;
  double ahead[kAhead][kItems];
  auto ask_values = [&](int first, int buf, int c, int n) {
    const uint16_t* index   = s_index + buf * a.chunk * R;
    const double* leaf_base = st.leaves + (static_cast<int64_t>(first) << a.depth) * a.K;
#pragma unroll
    for (int u = 0; u < kAhead; u++) {
      const int cc = min(c + u, n - 1);  // past the last tree: its value again, which is not added
#pragma unroll
      for (int i = 0; i < kItems; i++) {
        const uint32_t at = static_cast<uint32_t>((cc << a.depth) + index[cc * R + item_row[i]]) * a.K + item_out[i];
        ahead[u][i] = *reinterpret_cast<const double*>(reinterpret_cast<const char*>(leaf_base) + 8 * at);
      }
    }
  };
  auto add_values = [&](int c, int n) {
#pragma unroll
    for (int u = 0; u < kAhead; u++)
      if (c + u < n) {
#pragma unroll
        for (int i = 0; i < kItems; i++) acc[i] += ahead[u][i];
      }
  };
  auto add_rest = [&](int first, int buf, int n) {
    for (int c = kAhead; c < n; c += kAhead) {
      ask_values(first, buf, c, n);
      add_values(c, n);
    }
  };

  double val[kJ];
  int held = 0;  // kOwn: trees whose values are on their way
  auto add_held = [&]() {
    if (held == kJ) {
#pragma unroll
      for (int j = 0; j < kJ; j++) acc[0] += val[j];
    } else {
#pragma unroll
      for (int j = 0; j < kJ; j++)
        if (j < held) acc[0] += val[j];
    }
  };
  int buf = 0, turn = 0;
  for (int first = 0; first < a.n_trees; first += a.chunk, buf ^= 1) {
    const bool more = first + a.chunk < a.n_trees;
    if (more) fetch(first + a.chunk);
    const int before = min(a.chunk, a.n_trees - (first - a.chunk));
    const bool adds  = first > 0 && (kAdds == Adds::kShared || (kAdds == Adds::kInTurn && tw == turn));
    if (!kOwn && adds) ask_values(first - a.chunk, buf ^ 1, 0, before);
    const uint32_t nodes    = lds_base + a.node_off + (buf << (a.depth + 2)) * a.chunk;
    const uint32_t leaf_lds = lds_base + a.index_off + buf * n16_leaf * 16;
    for (int g = 0; g < per_wave; g += kJ) {
      const int t = tw * per_wave + g;
      uint32_t pos[kJ];
      walk_trees<kJ>(pos, nodes + (t << (a.depth + 2)), a.depth, lane_x, stride);
      if constexpr (kOwn) {
        // one turn per chunk: the next chunk's nodes are stored before this one's values are asked for, so that the
        // store does not wait for them (loads arrive in order)
        if (more) store(buf ^ 1);
        add_held();
        const char* leaf_base = reinterpret_cast<const char*>(st.leaves + (static_cast<int64_t>(first + t) << a.depth));
        held = min(kJ, a.n_trees - (first + t));
#pragma unroll
        for (int j = 0; j < kJ; j++)
          if (j < kLdsLeaves)
            val[j] = *lds_at<double>(8 * pos[j] + (leaf_lds + ((j - 1) << (a.depth + 3))));
          else
            val[j] = *reinterpret_cast<const double*>(leaf_base + (8 * pos[j] + ((j - 1) << (a.depth + 3))));
      } else {
#pragma unroll
        for (int j = 0; j < kJ; j++)
          s_index[(buf * a.chunk + t + j) * R + my_row] = static_cast<uint16_t>(pos[j] - (1 << a.depth));
      }
    }
    if constexpr (!kOwn) {
      if (adds) {
        if (kAdds == Adds::kInTurn) acc[0] = s_acc[my_row];
        add_values(0, before);
        add_rest(first - a.chunk, buf ^ 1, before);
        if (kAdds == Adds::kInTurn) s_acc[my_row] = acc[0];
      }
      if (first > 0) turn = turn + 1 == tree_waves ? 0 : turn + 1;
      if (more) store(buf ^ 1);
    }
    __syncthreads();
  }
  if constexpr (kOwn) {
    add_held();
    if (my_row < rows_here) out[row0 + my_row] = acc[0];
  } else {
    const int first = (a.n_trees - 1) / a.chunk * a.chunk, n = a.n_trees - first;
    if (kAdds == Adds::kInTurn) {
      if (tw != 0) return;
      acc[0] = s_acc[my_row];
    }
    ask_values(first, buf ^ 1, 0, n);
    add_values(0, n);
    add_rest(first, buf ^ 1, n);
    if constexpr (kAdds == Adds::kInTurn) {
      if (my_row < rows_here) out[row0 + my_row] = acc[0];
    } else {
#pragma unroll
      for (int i = 0; i < kItems; i++)
        if (lane + 64 * i < per_items && item_row[i] < rows_here) out[(row0 + item_row[i]) * a.K + item_out[i]] = acc[i];
    }
  }
}

struct Shape {
  int tile_rows = 0, chunk = 0, j = 0, items = 0;
  size_t lds = 0;
  int node_off = 0, index_off = 0, acc_off = 0;
};

// Rows of a tile and trees of a chunk for the LDS; tile_rows 0 when nothing fits.
Shape walk_shape(int64_t N, int F, int K, int depth)
{
  // several outputs: two workgroups per CU where they fit, one waits for leaf values while the other walks
  for (const size_t limit : {K > 1 ? kLds / 2 : kLds, kLds})
    for (int rows = 1024; rows >= 64; rows /= 2) {
      if (rows > 64 && N < static_cast<int64_t>(rows) * 512) continue;  // two tiles per CU at least
      const int tree_waves = kWalkThreads / rows;
      const bool own       = rows == 1024 && K == 1;
      const int items      = K == 1 ? 1 : (rows * K / kWalkWaves + 63) / 64;
      if (items > 2) continue;  // values on their way fill the registers
      const size_t x_bytes = static_cast<size_t>(rows) * F * 2;
      for (int per_wave = own || K == 1 ? 8 : 16; per_wave >= 1; per_wave /= 2) {
        const int chunk          = per_wave * tree_waves;
        const size_t node_bytes  = static_cast<size_t>(chunk) << (depth + 2);
        const size_t index_bytes = own ? (per_wave == 8 ? static_cast<size_t>(kLeavesInLds) << (depth + 3) : 0)
                                       : static_cast<size_t>(chunk) * rows * 2;
        const size_t acc_bytes   = K == 1 && !own ? static_cast<size_t>(rows) * 8 : 0;
        const size_t lds         = x_bytes + 2 * node_bytes + 2 * index_bytes + acc_bytes;
        if (lds > limit || node_bytes > static_cast<size_t>(kWalkCopy) * kWalkThreads * 16 || node_bytes % 16 != 0) continue;
        if (per_wave < (limit < kLds ? 1 : 4) && rows > 64) break;  // a smaller tile lets a wave walk more trees at once
        Shape s;
        s.tile_rows = rows;
        s.chunk     = chunk;
        s.j         = std::min(per_wave, 8);
        s.items     = own ? 0 : items;
        s.lds       = lds;
        s.node_off  = static_cast<int>(x_bytes);
        s.index_off = static_cast<int>(x_bytes + 2 * node_bytes);
        s.acc_off   = static_cast<int>(x_bytes + 2 * node_bytes + 2 * index_bytes);
        return s;
      }
    }
  return Shape{};
}

struct Plan {
  Shape shape;
  int depth = 0, padded_trees = 0, group = 0, cells = 0, rank_lds = 0;
  int turn_rows = 0;  // of features by the line
  int64_t slots = 0, thresholds = 0, chunk_rows = 0;
  bool may_overflow = false;
  size_t bytes = 0;
};

// Which way is the faster one, by costs (us) fitted to both over 250 shapes of 2000 to 4,000,000 rows, 4 to 500 features, 1 to
// 1000 trees of depth 3 to 8, 1 to 8 outputs and both types. By ranks: the launches that rank the thresholds, a pass
// over X that reads it and writes ranks (3.5 TB/s with its searches), node steps by how many trees a wave walks at once,
// the leaf rows of several outputs (twice as dear once the ensemble's exceed an XCD's L2). Tiled: X at 3.2 TB/s, node
// steps by the lanes a row takes and the share of a batch's trees that fits the LDS beside the rows, leaf rows. Rows that
// do not fit the LDS are walked in memory, 60,000 steps a microsecond. Since then a pass over X by the line and the packing of up to 64 trees became
// shorter: of 93 other shapes of these ranges ten that are tiled would be 6 to 69 % faster by ranks (1,101,139 x 9 f64, 13 trees of depth 8,
// 2 outputs 269 and 159 us), two that take ranks 3 % faster tiled. Examples, tiled against ranks: 2,410,724 x 53, 333
// trees of depth 7: 2702 and 1766 us; 2,087,561 x 104, 626 of depth 6: 5394 and 2736; 1,330,881 x 145 f64, 831 of depth 8:
// 31.5 and 4.35 ms; 65,071 x 54, 229 of depth 7: 91 and 201; 2,070,925 x 35, 16 of depth 5: 265 and 265.
bool ranks_are_faster(int64_t N, int F, int n_trees, int depth, int K, size_t value_size, const Shape& shape)
{
  const double rows = static_cast<double>(N), walks = rows * n_trees, steps = walks * depth;
  const double leaf_table = (static_cast<double>(n_trees) * K * 8.0) * (1u << depth);
  const double step_rate  = shape.items == 0 ? 4.5e6 : (shape.j >= 4 ? 3.5e6 : (shape.lds <= kLds / 2 ? 2.5e6 : 1.2e6));
  const double leaf_rows  = K > 1 ? walks * (1.0e-6 + 0.55e-6 * K) * (leaf_table > 3e6 ? 2.0 : 1.0) : 0.0;
  const double ranked     = 45.0 + 15.0 * ceil_div(n_trees, kPackTrees) + rows * F * (value_size + 4.0) / 3.5e6 +
                        steps / step_rate + leaf_rows;
  const size_t row_bytes = static_cast<size_t>(F | 1) * value_size;
  double walk            = std::max(steps / 0.06e6, 0.35 * n_trees * depth);
  const struct { int rows, trees; double f32, f64; } tiles[] = {{256, 20, 2.2e6, 1.5e6}, {128, 24, 1.45e6, 0.8e6}, {64, 32, 1.1e6, 0.6e6}};
  for (const auto& t : tiles) {
    const size_t x_bytes = row_bytes * t.rows;
    if (x_bytes > kLds * 55 / 100) continue;
    const double fit = static_cast<double>(kLds - x_bytes) / ((2u << depth) * 2.0 * value_size);
    walk = rows * F * value_size / 3.2e6 +
           steps / ((value_size == 4 ? t.f32 : t.f64) * std::min(1.0, fit / std::min(t.trees, n_trees)));
    break;
  }
  const double tiled = 10.0 + walk + (K > 1 ? 0.4e-6 * walks * std::pow(K, 1.4) : 0.0);
  return 1.05 * ranked < tiled;
}

Plan make_plan(int64_t N, int F, int n_trees, const int32_t* tree_nodes, int K, size_t value_size)
{
  Plan p;
  if (n_trees < 1 || F > 16383) return p;
  int64_t total = 0, thresholds = 0;
  int max_nodes = 0;
  for (int i = 0; i < n_trees; i++) {
    total += tree_nodes[i];
    thresholds += (tree_nodes[i] - 1) / 2;
    max_nodes = std::max(max_nodes, tree_nodes[i]);
  }
  while (((int64_t(1) << (p.depth + 1)) - 1) < max_nodes) p.depth++;
  if (p.depth < 1 || p.depth > 12) return p;
  const Shape s = walk_shape(N, F, K, p.depth);
  if (s.tile_rows == 0) return p;
  // a feature's thresholds beyond the sort's LDS are ranked by counting, which is slow (830 trees of depth 8 on four features: 9 ms)
  const int64_t sort_most = value_size == 4 ? kSortMost<float> : kSortMost<double>;
  if (thresholds > sort_most * F) return p;
  if (!ranks_are_faster(N, F, n_trees, p.depth, K, value_size, s)) return p;
  p.padded_trees = ceil_div(n_trees, s.chunk) * s.chunk;
  p.slots        = static_cast<int64_t>(p.padded_trees) << p.depth;
  if (p.slots > (int64_t(1) << 31) - 1 || p.slots > 2 * total + (static_cast<int64_t>(s.chunk) << p.depth)) return p;
  p.thresholds   = thresholds;
  p.may_overflow = thresholds > kMaxPerFeature;
  // rank workgroups: as many features as their thresholds fit the LDS, if they are spread evenly over the features
  const double mean = static_cast<double>(thresholds) / F;
  p.cells = 64;
  while (p.cells < 1024 && p.cells < 4 * mean) p.cells *= 2;
  auto bytes_for = [&](int group) {
    return (group * mean + 4.0 * std::sqrt(group * mean) + group) * static_cast<double>(value_size) + 2.0 * group * p.cells;
  };
  // the features of a 128-byte line if two such workgroups share a CU; else at most eight, in powers of two
  const int line = static_cast<int>(128 / value_size);
  if (F > kGroupMax && 2 * bytes_for(line) <= static_cast<double>(kLds / 2 - 1024)) {
    p.group     = line;
    p.turn_rows = 256;
  } else {
    p.group = 1;
    while (p.group < kGroupMax && p.group < F && bytes_for(2 * p.group) <= static_cast<double>(kLds - 1024)) p.group *= 2;
  }
  // what all thresholds on these features would take, or room for twice the mean; of a line as much as is left beside the turned rows. Turns of
  // doubles are half as long where such a line would not have that with few cells: 63,232 bytes instead of 46,592 (2,000,000 x 100, 50 trees of depth 8, of
  // which a share of 0.45 on one line 969 us; 1794 searched in memory, as with whole turns. 300,000 rows, evenly: 203 and 200)
  const double twice = 2.0 * bytes_for(p.group);
  double room        = std::max(twice, 32.0 * 1024), most_room = static_cast<double>(kLds - 1024);
  if (p.group == line) {
    most_room = static_cast<double>(kLds / 2 - 1024 - line_stage(value_size, p.turn_rows));
    if (value_size == 8 && twice - 2.0 * line * (p.cells - kFewCells) > most_room) {
      p.turn_rows = 128;
      most_room   = static_cast<double>(kLds / 2 - 1024 - line_stage(value_size, p.turn_rows));
    }
    room = most_room;
  }
  const double all_here = (static_cast<double>(thresholds) + 1) * static_cast<double>(value_size) + 2.0 * p.group * p.cells;
  p.rank_lds = static_cast<int>(std::min(std::min(all_here, room) + 15, most_room)) / 16 * 16;
  const int64_t tiles = (N + s.tile_rows - 1) / s.tile_rows;
  const int64_t most  = std::max<int64_t>(256, static_cast<int64_t>(kRankedChunkBytes / (static_cast<size_t>(s.tile_rows) * F * 2)) / 256 * 256);
  p.chunk_rows = std::min(tiles, most) * s.tile_rows;
  p.shape      = s;
  return p;
}

template <typename T>
struct Layout {
  RankState st{};
  T *raw, *grouped, *sorted;
  uint16_t* ranks;
  size_t bytes;
  Layout(void* buffer, const Plan& p, int F, int K)
  {
    Arena ar;
    ar.measure = buffer == nullptr;
    ar.base    = reinterpret_cast<char*>((reinterpret_cast<uintptr_t>(buffer) + 255) & ~uintptr_t(255));
    ar.cap     = ~size_t(0);
    st.depth   = p.depth;
    st.F       = F;
    st.K       = K;
    st.n_trees = p.padded_trees;
    st.count    = ar.take<int32_t>(2 * static_cast<int64_t>(F));
    st.offset   = ar.take<int32_t>(F + 1);
    st.overflow = ar.take<int32_t>(1);
    st.slot     = ar.take<uint32_t>(p.slots);
    st.nodes    = ar.take<uint32_t>(p.slots);
    st.leaves   = ar.take<double>(p.slots * K);
    st.owner    = ar.take<uint32_t>(p.thresholds + 1);
    raw         = ar.take<T>(p.slots);
    grouped     = ar.take<T>(p.thresholds + 1);
    sorted      = ar.take<T>(p.thresholds + 1);
    ranks       = ar.take<uint16_t>(p.chunk_rows * F);
    bytes       = ar.used + 512;
  }
};

template <typename T>
size_t ranked_bytes(const Plan& p, int F, int K)
{
  return Layout<T>(nullptr, p, F, K).bytes;
}

}  // namespace

size_t ranked_workspace_bytes(int64_t N, int F, int n_trees, const int32_t* tree_nodes, int K, int x_dtype)
{
  const Plan p = make_plan(N, F, n_trees, tree_nodes, K, x_dtype == LBT_F32 ? 4 : 8);
  if (p.shape.tile_rows == 0) return 0;
  return x_dtype == LBT_F32 ? ranked_bytes<float>(p, F, K) : ranked_bytes<double>(p, F, K);
}

template <typename T>
int predict_ranked(hipStream_t stream, const T* X, int64_t N, int F, int n_trees, const double* const* leaf,
                   const int32_t* const* feature, const double* const* split, const int32_t* tree_nodes, int K,
                   double* out, void* workspace, size_t workspace_bytes, bool* done, const int32_t** overflow)
{
  *done     = false;
  *overflow = nullptr;
  const Plan p = make_plan(N, F, n_trees, tree_nodes, K, sizeof(T));
  if (p.shape.tile_rows == 0 || workspace == nullptr || workspace_bytes < ranked_bytes<T>(p, F, K)) return LBT_OK;
  Layout<T> lay(workspace, p, F, K);
  RankState& st = lay.st;
  ProfScope ps(LBT_PROF_PREDICT, stream, static_cast<double>(N) * (static_cast<double>(F) * sizeof(T) + K * 8.0));
  zero_counts_kernel<<<ceil_div(2 * F, kThreads), kThreads, 0, stream>>>(st.count, 2 * F);
  for (int first = 0; first < p.padded_trees; first += kPackTrees) {
    PackRefs refs{};
    const int all  = std::min(kPackTrees, p.padded_trees - first);
    const int here = std::max(0, std::min(kPackTrees, n_trees - first));
    for (int i = 0; i < here; i++) {
      refs.leaf[i]    = leaf[first + i];
      refs.feature[i] = feature[first + i];
      refs.split[i]   = split[first + i];
      refs.n_nodes[i] = tree_nodes[first + i];
    }
    // few trees: one to a workgroup, whose chain of loads is what the launch lasts (50 trees with 8 outputs 24 us by fours, 8 alone)
    auto pack = [&](auto together) {
      constexpr int kTogether = decltype(together)::value;
      const dim3 grid(ceil_div(1 << p.depth, kThreads), ceil_div(all, kTogether));
      if (F <= kLocalCounters)
        rank_pack_kernel<T, true, kTogether><<<grid, kThreads, F * sizeof(int32_t), stream>>>(refs, first, here, all, st, lay.raw);
      else
        rank_pack_kernel<T, false, kTogether><<<grid, kThreads, 0, stream>>>(refs, first, here, all, st, lay.raw);
    };
    if (p.padded_trees <= 64)
      pack(std::integral_constant<int, 1>{});
    else
      pack(std::integral_constant<int, kPackTogether>{});
  }
  rank_offsets_kernel<<<1, 1024, 0, stream>>>(st);
  rank_scatter_kernel<T><<<ceil_div(p.slots, kThreads), kThreads, 0, stream>>>(st, lay.raw, lay.grouped);
  static std::atomic<bool> sort_attr[kMaxDevices] = {};
  const size_t sort_most = std::min<size_t>(kSortMost<T>, static_cast<size_t>(p.thresholds));
  size_t sort_size       = kRankTile;
  while (sort_size < sort_most) sort_size *= 2;
  LBT_TRY(allow_dynamic_lds(rank_thresholds_kernel<T>, kSortMost<T> * (sizeof(T) + sizeof(uint32_t)), sort_attr));
  rank_thresholds_kernel<T><<<dim3(F, p.thresholds > kSortMost<T> ? kRankBlocks : 1), kSortThreads,
                              sort_size * (sizeof(T) + sizeof(uint32_t)), stream>>>(st, static_cast<int>(sort_size), lay.grouped, lay.sorted);

  static std::atomic<bool> rank_attr[6][kMaxDevices] = {};
  static std::atomic<bool> walk_attr[4][4][kMaxDevices] = {};
  auto whole_words = [&](const T* x) { return (static_cast<size_t>(F) * sizeof(T)) % 16 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0; };
  // features of a workgroup; rows of a turn where they are those of a line, else 0
  auto rank_chunk = [&](auto group_c, auto turn_c, std::atomic<bool> (&flags)[kMaxDevices], const T* x, int64_t rows) -> int {
    constexpr int kG = decltype(group_c)::value, kTurn = decltype(turn_c)::value;
    constexpr bool kLine = kTurn > 0;
    if constexpr (kLine)
      LBT_TRY((allow_dynamic_lds(rank_lines_kernel<T, kTurn>, kLds - 1024, flags)));
    else
      LBT_TRY((allow_dynamic_lds(rank_rows_kernel<T, kG>, kLds - 1024, flags)));
    RankRows a{};
    a.n_rows    = rows;
    a.F         = F;
    a.n_groups  = ceil_div(F, kG);
    a.tile_shift = 31 - __builtin_clz(static_cast<unsigned>(p.shape.tile_rows));
    a.cells     = p.cells;
    a.lds_bytes = p.rank_lds;
    // row ranges in multiples of the XCDs, as many as run at once
    const size_t lds     = p.rank_lds + (kLine ? line_stage(sizeof(T), kTurn) : 0);
    const int per_cu     = kLds / 2 >= lds + 1024 ? 2 : 1;
    const int64_t splits = 8 * std::max<int64_t>(1, std::min<int64_t>(32 * per_cu / a.n_groups, ceil_div(rows, 8 * kWalkThreads)));
    a.rows_per_split     = (rows + splits * kWalkThreads - 1) / (splits * kWalkThreads) * kWalkThreads;
    a.wide = whole_words(x) && kG * sizeof(T) >= 16;
    const unsigned grid = static_cast<unsigned>(splits * a.n_groups);
    if constexpr (kLine)
      rank_lines_kernel<T, kTurn><<<grid, kWalkThreads, lds, stream>>>(x, a, st, lay.sorted, lay.ranks);
    else
      rank_rows_kernel<T, kG><<<grid, kWalkThreads, lds, stream>>>(x, a, st, lay.sorted, lay.ranks);
    return LBT_OK;
  };
  auto walk_chunk = [&](auto adds_c, auto items_c, auto j_c, std::atomic<bool> (&flags)[kMaxDevices], int64_t rows, double* o) -> int {
    constexpr Adds kA = decltype(adds_c)::value;
    constexpr int kI = decltype(items_c)::value, kJ = decltype(j_c)::value;
    LBT_TRY((allow_dynamic_lds(walk_ranked_kernel<kA, kI, kJ>, kLds, flags)));
    WalkArgs a{};
    a.n_rows    = rows;
    a.F         = F;
    a.K         = K;
    a.depth     = p.depth;
    a.n_trees   = n_trees;
    a.tile_rows = p.shape.tile_rows;
    a.chunk     = p.shape.chunk;
    a.node_off  = p.shape.node_off;
    a.index_off = p.shape.index_off;
    a.acc_off   = p.shape.acc_off;
    walk_ranked_kernel<kA, kI, kJ><<<ceil_div(rows, a.tile_rows), kWalkThreads, p.shape.lds, stream>>>(lay.ranks, a, st, o);
    return LBT_OK;
  };
  using std::integral_constant;
  for (int64_t row = 0; row < N; row += p.chunk_rows) {
    const int64_t rows = std::min(p.chunk_rows, N - row);
    const T* x = X + row * F;
    double* o  = out + row * K;
    const integral_constant<int, 1> one{};
    const integral_constant<int, 0> none{};
    switch (p.group) {
      case 1: LBT_TRY(rank_chunk(one, none, rank_attr[0], x, rows)); break;
      case 2: LBT_TRY(rank_chunk(integral_constant<int, 2>{}, none, rank_attr[1], x, rows)); break;
      case 4: LBT_TRY(rank_chunk(integral_constant<int, 4>{}, none, rank_attr[2], x, rows)); break;
      case 8: LBT_TRY(rank_chunk(integral_constant<int, 8>{}, none, rank_attr[3], x, rows)); break;
      default:
        if (p.turn_rows == 256)
          LBT_TRY(rank_chunk(integral_constant<int, kLineFeatures<T>>{}, integral_constant<int, 256>{}, rank_attr[4], x, rows));
        else if constexpr (sizeof(T) == 8)
          LBT_TRY(rank_chunk(integral_constant<int, kLineFeatures<T>>{}, integral_constant<int, 128>{}, rank_attr[5], x, rows));
        break;
    }
    auto with = [&](auto adds_c, auto items_c, int at) -> int {
      switch (p.shape.j) {
        case 1: return walk_chunk(adds_c, items_c, integral_constant<int, 1>{}, walk_attr[0][at], rows, o);
        case 2: return walk_chunk(adds_c, items_c, integral_constant<int, 2>{}, walk_attr[1][at], rows, o);
        case 4: return walk_chunk(adds_c, items_c, integral_constant<int, 4>{}, walk_attr[2][at], rows, o);
        default: return walk_chunk(adds_c, items_c, integral_constant<int, 8>{}, walk_attr[3][at], rows, o);
      }
    };
    if (p.shape.items == 0)
      LBT_TRY(with(integral_constant<Adds, Adds::kOwn>{}, one, 0));
    else if (K == 1)
      LBT_TRY(with(integral_constant<Adds, Adds::kInTurn>{}, one, 1));
    else if (p.shape.items == 1)
      LBT_TRY(with(integral_constant<Adds, Adds::kShared>{}, one, 2));
    else
      LBT_TRY(with(integral_constant<Adds, Adds::kShared>{}, integral_constant<int, 2>{}, 3));
  }
  LBT_HIP(hipGetLastError());
  *done = true;
  if (p.may_overflow) *overflow = st.overflow;
  return LBT_OK;
}

template int predict_ranked<float>(hipStream_t, const float*, int64_t, int, int, const double* const*, const int32_t* const*,
                                   const double* const*, const int32_t*, int, double*, void*, size_t, bool*, const int32_t**);
template int predict_ranked<double>(hipStream_t, const double*, int64_t, int, int, const double* const*, const int32_t* const*,
                                    const double* const*, const int32_t*, int, double*, void*, size_t, bool*, const int32_t**);

}  // namespace lbt
