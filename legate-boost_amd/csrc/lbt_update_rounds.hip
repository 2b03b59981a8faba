// LBBase.update (legateboost/legateboost.py:306-386) over the trees of a fitted model: per tree the weighted gradient at the
// predictions so far, UpdateTreeTask (src/models/tree/update_tree.cc:36-122) and the prediction update.
//
// Only the sums of a tree depend on the trees before it; where the rows stop does not. So X is read once for many
// trees (tree_leaves_kernel) and a round is one pass over the targets and predictions (round_kernel), which adds the leaf
// values of the tree before, forms gradient and hessian and sums them per node. Inner nodes and outputs of all
// trees follow at the end. One tree after the other (gradient, accumulation over X, finish, prediction update) took
// 82 us a tree on 1,000,000 x 50 with depth 8, of which 59 were for X; now 61 for ten trees and 8 a round.
#include <algorithm>
#include <type_traits>

#include "lbt_internal.h"
#include "lbt_trees.h"

namespace lbt {
namespace {

constexpr int kPassTrees     = 16;          // trees whose nodes lie in the LDS at a time
constexpr int kLeafThreads   = 512;
constexpr int kRoundThreads  = 1024;
constexpr int kTogether      = 4;           // trees a lane walks at once, at most
constexpr int kAheadWords    = 8;           // 16-byte words of the next tile that a lane holds
constexpr size_t kNodeLds    = 64 * 1024;
constexpr size_t kTwoPerCu   = 78 * 1024;
constexpr size_t kOnePerCu   = 158 * 1024;
constexpr int kMostSums      = 4096;        // nodes * outputs of a tree: two sums and the leaf values of one before in the LDS
constexpr int kPackTrees     = 32;          // descriptors passed by value per launch
constexpr size_t kLeafBytes  = 128u << 20;  // recorded leaves of one pass
constexpr int kCopies        = 8;           // of a tree's sums: a workgroup adds to one of them
constexpr int kLaneCopies    = 4;           // of the sums in a workgroup's LDS, where kCopiesLds holds them: rows of one node meet less often
constexpr size_t kCopiesLds  = 64 * 1024;
constexpr int kStagedPerStep = 80;          // a scattered cache line costs as much as about 100 bytes in sequence

struct PackRefs {
  const int32_t* feature[kPackTrees];
  const double* split[kPackTrees];
  int64_t node_off[kPackTrees];
  int32_t n_nodes[kPackTrees];
};

// n trees, a row of workgroups each; the row behind them clears the sums
template <typename T>
__global__ void __launch_bounds__(256) pack_update_nodes_kernel(PackRefs refs, int n, int F, PackedNode<T>* nodes, double* sums, int64_t n_sums)
{
  const int t = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
  if (t == n) {
    for (int64_t s = i; s < n_sums; s += static_cast<int64_t>(gridDim.x) * 256) sums[s] = 0.0;
    return;
  }
  if (i < refs.n_nodes[t]) nodes[refs.node_off[t] + i] = pack_node<T>(i, refs.feature[t][i], refs.split[t][i], F, refs.n_nodes[t]);
}

struct LeavesArgs {
  int64_t n_rows, n_tiles;
  int F, pitch, tile_rows, n_trees, steps;
  int node_words;  // 16-byte words of the trees' nodes
  int node_off[kPassTrees];
};

typedef unsigned int Word16 __attribute__((ext_vector_type(4)));

// The node every row stops in, for up to kPassTrees trees. Their nodes stay in the LDS; kStaged: so do the rows of a tile, whose
// successor is on its way into registers meanwhile (rows too wide for that are walked in memory). The lanes of a row take its
// trees in turn, kWalks each side by side. What bounds it are the walk's LDS reads, two a step and lane: walks that no tree needs are as dear as
// others (1,000,000 x 50, 10 trees of depth 8, four lanes a row: with four walks each 61 us, with three 55).
template <typename T, bool kStaged, int kWalks>
__global__ void __launch_bounds__(kLeafThreads)
  tree_leaves_kernel(const T* __restrict__ X, LeavesArgs a, const PackedNode<T>* __restrict__ nodes, uint16_t* __restrict__ row_leaf)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const PackedNode<T>* s_nodes = reinterpret_cast<const PackedNode<T>*>(smem_raw);
  T* s_x        = reinterpret_cast<T*>(smem_raw + static_cast<size_t>(a.node_words) * 16);
  const int tid = threadIdx.x;
  for (int i = tid; i < a.node_words; i += kLeafThreads)
    reinterpret_cast<Word16*>(smem_raw)[i] = reinterpret_cast<const Word16*>(nodes)[i];
  const int r = tid & (a.tile_rows - 1), q = tid / a.tile_rows, lanes = kLeafThreads / a.tile_rows;
  constexpr int kPer = 16 / sizeof(T);
  // a tile starts on a 16-byte boundary when X does: its rows are a multiple of 64
  const bool words = (reinterpret_cast<uintptr_t>(X) & 15) == 0;
  Word16 ahead[kAheadWords];
  auto elements = [&](int64_t tile) {
    return static_cast<int>(min<int64_t>(a.tile_rows, a.n_rows - tile * a.tile_rows)) * a.F;
  };
  auto fetch = [&](int64_t tile) {
    const Word16* src = reinterpret_cast<const Word16*>(X + tile * a.tile_rows * a.F);
    const int n       = elements(tile) / kPer;
#pragma unroll
    for (int c = 0; c < kAheadWords; c++)
      if (tid + c * kLeafThreads < n) ahead[c] = src[tid + c * kLeafThreads];
  };
  auto put = [&](int e, T v) {
    // rows of whole words are set apart by one value, so that a column lies in many banks; others lie end to end
    s_x[a.pitch == a.F ? e : e / a.F * a.pitch + e % a.F] = v;
  };
  auto stage = [&](int64_t tile) {
    const T* src    = X + tile * a.tile_rows * a.F;
    const int total = elements(tile), n = words ? total / kPer : 0;
    auto put_word   = [&](int i, const Word16& w) {
      if (a.pitch == a.F) {
        reinterpret_cast<Word16*>(s_x)[i] = w;
      } else {
        T v[kPer];
        __builtin_memcpy(v, &w, 16);
        const int row = i / (a.F / kPer);
        T* d          = s_x + row * a.pitch + (i - row * (a.F / kPer)) * kPer;
#pragma unroll
        for (int j = 0; j < kPer; j++) d[j] = v[j];
      }
    };
    if (words) {
#pragma unroll
      for (int c = 0; c < kAheadWords; c++)
        if (tid + c * kLeafThreads < n) put_word(tid + c * kLeafThreads, ahead[c]);
      for (int i = tid + kAheadWords * kLeafThreads; i < n; i += kLeafThreads)
        put_word(i, reinterpret_cast<const Word16*>(src)[i]);
    }
    for (int e = n * kPer + tid; e < total; e += kLeafThreads) put(e, src[e]);
  };
  if (kStaged && words && blockIdx.x < a.n_tiles) fetch(blockIdx.x);
  for (int64_t tile = blockIdx.x; tile < a.n_tiles; tile += gridDim.x) {
    if constexpr (kStaged) {
      __syncthreads();  // the tile before is no longer read
      stage(tile);
    }
    __syncthreads();
    if (kStaged && words && tile + gridDim.x < a.n_tiles) fetch(tile + gridDim.x);
    const int64_t row = tile * a.tile_rows + r;
    const bool valid  = row < a.n_rows;
    const T* x        = kStaged ? s_x + (valid ? r : 0) * a.pitch : X + (valid ? row : 0) * a.F;
    for (int t0 = q; t0 < a.n_trees; t0 += kWalks * lanes) {
      int base[kWalks], pos[kWalks];
#pragma unroll
      for (int j = 0; j < kWalks; j++) {
        base[j] = a.node_off[min(t0 + j * lanes, a.n_trees - 1)];
        pos[j]  = 0;
      }
      for (int s = 0; s < a.steps; s++) {
#pragma unroll
        for (int j = 0; j < kWalks; j++) pos[j] = step_from<T>(s_nodes[base[j] + pos[j]], x);
      }
#pragma unroll
      for (int j = 0; j < kWalks; j++)
        if (valid && t0 + j * lanes < a.n_trees)
          row_leaf[static_cast<int64_t>(t0 + j * lanes) * a.n_rows + row] = static_cast<uint16_t>(pos[j]);
    }
  }
}

struct RoundArgs {
  int64_t n_rows;
  int K, n_nodes, prev_nodes;  // prev_nodes: 0 in the first round
  int lane_copies;             // of the sums in the LDS, a power of two
  double lr;
  const double* y;
  const double* weight;
  double* pred;
  const uint16_t* leaf;       // node of every row in this round's tree
  const uint16_t* prev_leaf;  // and in the one before
  const double* prev_sums;    // its sums, as below
  double prev_l1, prev_l2;
  double* sums;               // [kCopies][2][n_nodes][K]
};

// sums of gradients (which 0) or hessians (1) at entry i of n
__device__ __forceinline__ double sum_of_copies(const double* sums, int n, int which, int i)
{
  double v = 0.0;
#pragma unroll
  for (int c = 0; c < kCopies; c++) v += sums[static_cast<int64_t>(2 * c + which) * n + i];
  return v;
}

enum class Gradient { kSquared, kLogistic, kSoftmax };

// One round (see above): the leaf values of the tree before are formed by every workgroup from its sums, so nothing runs
// between two rounds. The gradient is lbt_weighted_gradient's, operation by operation. kCols: the outputs where
// they are known (1, or a softmax row in registers), 0 any number.
// kCounts: squared errors of rows without weights, whose hessians are ones: they are counted (a 32-bit add of the LDS for one of 64 bits).
// What bounds it, 1,000,000 rows and trees of depth 8: 4.4 us are the launch and its barriers, 1.8 the workgroups' adds to the sums in memory
// (one address takes them in turn: with one copy of the sums 256 workgroups took 13.2 us in all; of 4, 8, 16 and 32 copies 8 are best), 1.2 each the sums of the
// tree before and the rows, the rest the adds in the LDS (rows apart by lanes in kLaneCopies: 9.05 -> 8.5 us a launch, counts: 8.2).
template <Gradient kKind, int kCols, bool kCounts>
__global__ void __launch_bounds__(kRoundThreads) round_kernel(RoundArgs a)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int K = kCols > 0 ? kCols : a.K, n_sums = a.n_nodes * K, n_prev = a.prev_nodes * K, tid = threadIdx.x;
  double* s_prev = reinterpret_cast<double*>(smem_raw);  // [prev_nodes][K]
  double* s_sum  = s_prev + n_prev;                      // [lane_copies][2][K][n_nodes]: nodes side by side in the banks
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kRoundThreads;
  const int64_t first  = blockIdx.x * static_cast<int64_t>(kRoundThreads) + tid;
  // one output: the values of the next kRows rows of a thread; the first ones are asked for before the sums of the tree before
  constexpr int kRows = 4;
  double p_next[kRows], y_next[kRows], w_next[kRows];
  int node_next[kRows], prev_next[kRows];
  auto fetch = [&](int64_t row0) {
#pragma unroll
    for (int u = 0; u < kRows; u++) {
      const int64_t row = min(row0 + u * stride, a.n_rows - 1);
      p_next[u]    = a.pred[row];
      y_next[u]    = a.y[row];
      w_next[u]    = a.weight != nullptr ? a.weight[row] : 1.0;
      node_next[u] = a.leaf[row];
      prev_next[u] = n_prev > 0 ? a.prev_leaf[row] : 0;
    }
  };
  if constexpr (kCols == 1) fetch(first);
  for (int i = tid; i < n_prev; i += kRoundThreads)
    s_prev[i] = updated_leaf(sum_of_copies(a.prev_sums, n_prev, 0, i), sum_of_copies(a.prev_sums, n_prev, 1, i), a.prev_l1, a.prev_l2);
  for (int i = tid; i < 2 * n_sums * a.lane_copies; i += kRoundThreads) s_sum[i] = 0.0;
  __syncthreads();
  double* const own_sum = s_sum + (tid & (a.lane_copies - 1)) * 2 * n_sums;
  auto add = [&](int node, int k, double g, double h) {
    unsafeAtomicAdd(&own_sum[k * a.n_nodes + node], g);
    if constexpr (kCounts)
      atomicAdd(reinterpret_cast<uint32_t*>(own_sum + n_sums) + (k * a.n_nodes + node), 1u);
    else
      unsafeAtomicAdd(&own_sum[n_sums + k * a.n_nodes + node], h);
  };
  if constexpr (kCols == 1) {
    for (int64_t row0 = first; row0 < a.n_rows; row0 += kRows * stride) {
      double p[kRows], y[kRows], w[kRows];
      int node[kRows], prev[kRows];
#pragma unroll
      for (int u = 0; u < kRows; u++) {
        p[u]    = p_next[u];
        y[u]    = y_next[u];
        w[u]    = w_next[u];
        node[u] = node_next[u];
        prev[u] = prev_next[u];
      }
      if (row0 + kRows * stride < a.n_rows) fetch(row0 + kRows * stride);
#pragma unroll
      for (int u = 0; u < kRows; u++) {
        const int64_t row = row0 + u * stride;
        if (row >= a.n_rows) break;
        if (n_prev > 0) {
          p[u] += s_prev[prev[u]];
          a.pred[row] = p[u];
        }
        double h0 = 1.0, q = p[u], g, h;
        if constexpr (kKind == Gradient::kLogistic) {
          q  = 1.0 / (1.0 + exp(-q));
          h0 = q * (1.0 - q);
        }
        weigh(q - y[u], h0, w[u], a.lr, &g, &h);
        add(node[u], 0, g, h);
      }
    }
  } else {
    for (int64_t row = first; row < a.n_rows; row += stride) {
      const double w     = a.weight != nullptr ? a.weight[row] : 1.0;
      const int node     = a.leaf[row];
      const double* leaf = s_prev + (n_prev > 0 ? a.prev_leaf[row] * K : 0);
      double* p          = a.pred + row * K;
      auto current       = [&](int k) {
        if (n_prev == 0) return p[k];
        const double v = p[k] + leaf[k];
        p[k]           = v;
        return v;
      };
      double g, h;
      if constexpr (kKind == Gradient::kSquared) {
        for (int k = 0; k < K; k++) {
          weigh(current(k) - a.y[row * K + k], 1.0, w, a.lr, &g, &h);
          add(node, k, g, h);
        }
      } else {
        const int label = static_cast<int>(a.y[row]);
        auto take       = [&](int k, double q) {
          weigh(k == label ? q + -1.0 : q, q * (1.0 - q), w, a.lr, &g, &h);
          add(node, k, g, h);
        };
        if constexpr (kCols > 0) {
          double e[kCols];
#pragma unroll
          for (int k = 0; k < kCols; k++) e[k] = current(k);
          double top = e[0];
#pragma unroll
          for (int k = 0; k < kCols; k++) top = fmax(top, e[k]);
          double div = 0.0;
#pragma unroll
          for (int k = 0; k < kCols; k++) {
            e[k] = exp(e[k] - top);
            div += e[k];
          }
#pragma unroll
          for (int k = 0; k < kCols; k++) take(k, e[k] / div);
        } else {
          double top = current(0);
          for (int k = 1; k < K; k++) top = fmax(top, current(k));
          double div = 0.0;
          for (int k = 0; k < K; k++) div += exp(p[k] - top);
          for (int k = 0; k < K; k++) take(k, exp(p[k] - top) / div);
        }
      }
    }
  }
  __syncthreads();
  double* to = a.sums + static_cast<int64_t>(2) * n_sums * (blockIdx.x % kCopies);
  for (int i = tid; i < n_sums; i += kRoundThreads) {
    const int node = i / K, at = (i - node * K) * a.n_nodes + node;
    auto hess_at = [&](int c) {
      const double* h = s_sum + 2 * n_sums * c + n_sums;
      if constexpr (kCounts) return static_cast<double>(reinterpret_cast<const uint32_t*>(h)[at]);
      return h[at];
    };
    double gv = s_sum[at], hv = hess_at(0);
    for (int c = 1; c < a.lane_copies; c++) {
      gv += s_sum[2 * n_sums * c + at];
      hv += hess_at(c);
    }
    if (gv != 0.0) unsafeAtomicAdd(&to[i], gv);
    if (hv != 0.0) unsafeAtomicAdd(&to[n_sums + i], hv);
  }
}

struct FinishRefs {
  const int32_t* feature[kPackTrees];
  const double* sums[kPackTrees];  // [kCopies][2][n_nodes][K]
  double* leaf[kPackTrees];
  double* hessian[kPackTrees];
  double l1[kPackTrees], l2[kPackTrees];
  int32_t n_nodes[kPackTrees];
};

// Sums of inner nodes, leaf values and hessians: a workgroup per tree. The workgroups behind them add the last of these trees' values to the
// predictions: they form them from the sums, as a round does, and wait for no other launch (8.4 us and 6.2 behind it as two
// launches on 1,000,000 rows with ten trees, one of 11.9).
__global__ void __launch_bounds__(1024)
  finish_trees_kernel(FinishRefs refs, int n_trees, int K, const uint16_t* __restrict__ row_leaf, int64_t n_pred, double* pred)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int t = min(static_cast<int>(blockIdx.x), n_trees - 1), n = refs.n_nodes[t] * K;
  double* g   = reinterpret_cast<double*>(smem_raw);
  if (static_cast<int>(blockIdx.x) >= n_trees) {
    constexpr int kEntries = 4;
    const int64_t stride   = static_cast<int64_t>(gridDim.x - n_trees) * 1024;
    const int64_t first    = static_cast<int64_t>(blockIdx.x - n_trees) * 1024 + threadIdx.x;
    double p[kEntries];
    int at[kEntries];
    auto fetch = [&](int64_t i0) {
#pragma unroll
      for (int u = 0; u < kEntries; u++) {
        const int64_t i = min(i0 + u * stride, n_pred - 1), r = K == 1 ? i : i / K;
        at[u] = row_leaf[r] * K + static_cast<int>(i - r * K);
        p[u]  = pred[i];
      }
    };
    fetch(first);
    for (int i = threadIdx.x; i < n; i += 1024)
      g[i] = updated_leaf(sum_of_copies(refs.sums[t], n, 0, i), sum_of_copies(refs.sums[t], n, 1, i), refs.l1[t], refs.l2[t]);
    __syncthreads();
    for (int64_t i0 = first; i0 < n_pred; i0 += kEntries * stride) {
#pragma unroll
      for (int u = 0; u < kEntries; u++)
        if (i0 + u * stride < n_pred) pred[i0 + u * stride] = p[u] + g[at[u]];
      if (i0 + kEntries * stride < n_pred) fetch(i0 + kEntries * stride);
    }
    return;
  }
  double* h   = g + n;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    g[i] = sum_of_copies(refs.sums[t], n, 0, i);
    h[i] = sum_of_copies(refs.sums[t], n, 1, i);
  }
  __syncthreads();
  sum_inner_nodes(refs.feature[t], refs.n_nodes[t], K, g, h);
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    refs.leaf[t][i]    = updated_leaf(g[i], h[i], refs.l1[t], refs.l2[t]);
    refs.hessian[t][i] = h[i];
  }
}

int depth_of(int n_nodes)
{
  int depth = 0;
  while (((int64_t(1) << (depth + 1)) - 1) < n_nodes) depth++;
  return depth;
}

struct Plan {
  bool taken = false;
  int pass_trees = 0;
  int64_t nodes = 0, sums = 0;
  size_t bytes = 0;
};

Plan make_plan(int64_t N, int F, size_t value_size, int K, int n_trees, const int32_t* tree_nodes)
{
  Plan p;
  if (N < 1 || F > kMaxPackedFeatures || n_trees < 1) return p;
  for (int t = 0; t < n_trees; t++) {
    // whole levels, and sums that fit the LDS; other trees are updated one at a time
    if (tree_nodes[t] != (int64_t(1) << (depth_of(tree_nodes[t]) + 1)) - 1) return p;
    if (static_cast<int64_t>(tree_nodes[t]) * K > kMostSums) return p;
    if (static_cast<size_t>(tree_nodes[t] + 1) * 2 * value_size > kNodeLds) return p;
    p.nodes += tree_nodes[t] + 1;  // an even number: trees begin on 16 bytes
    p.sums += static_cast<int64_t>(2 * kCopies) * tree_nodes[t] * K;
  }
  p.pass_trees = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>({kPassTrees, n_trees, static_cast<int64_t>(kLeafBytes / 2) / N})));
  const int64_t held = std::min<int64_t>(n_trees, 2 * p.pass_trees);  // the round before may be the last of the pass before
  auto pad = [](size_t b) { return (b + 255) & ~size_t(255); };
  p.bytes  = pad(p.nodes * 2 * value_size) + pad(p.sums * sizeof(double)) + pad(static_cast<size_t>(held) * N * 2) + 512;
  p.taken  = true;
  return p;
}

template <typename T>
int update_rounds(hipStream_t stream, const T* X, int64_t N, int F, int objective, const double* y, const double* weight, double lr,
                  int K, int n_trees, const int32_t* const* feature, const double* const* split, const int32_t* tree_nodes,
                  const double* l1, const double* l2, double* pred, double* const* leaf_out, double* const* hessian_out,
                  void* workspace, const Plan& p)
{
  Arena ar;
  ar.base = reinterpret_cast<char*>((reinterpret_cast<uintptr_t>(workspace) + 255) & ~uintptr_t(255));
  ar.cap  = ~size_t(0);
  PackedNode<T>* nodes = ar.take<PackedNode<T>>(p.nodes);
  double* sums         = ar.take<double>(p.sums);
  uint16_t* row_leaf   = ar.take<uint16_t>(std::min<int64_t>(n_trees, 2 * p.pass_trees) * N);
  std::vector<int64_t> node_off(n_trees + 1, 0), sum_off(n_trees + 1, 0);
  for (int t = 0; t < n_trees; t++) {
    node_off[t + 1] = node_off[t] + tree_nodes[t] + 1;
    sum_off[t + 1]  = sum_off[t] + static_cast<int64_t>(2 * kCopies) * tree_nodes[t] * K;
  }
  for (int first = 0; first < n_trees; first += kPackTrees) {
    PackRefs refs{};
    const int n = std::min(kPackTrees, n_trees - first);
    int widest  = 1;
    for (int i = 0; i < n; i++) {
      refs.feature[i]  = feature[first + i];
      refs.split[i]    = split[first + i];
      refs.node_off[i] = node_off[first + i];
      refs.n_nodes[i]  = tree_nodes[first + i];
      widest           = std::max(widest, tree_nodes[first + i]);
    }
    const bool clears = first == 0;
    const int wide    = clears ? std::max<int>(ceil_div(widest, 256), static_cast<int>(std::min<int64_t>(256, ceil_div(p.sums, 2048)))) : ceil_div(widest, 256);
    pack_update_nodes_kernel<T><<<dim3(wide, n + (clears ? 1 : 0)), 256, 0, stream>>>(refs, n, F, nodes, sums, p.sums);
  }

  static std::atomic<bool> round_attr[15][kMaxDevices] = {}, finish_attr[kMaxDevices] = {};
  const unsigned round_grid = static_cast<unsigned>(std::min<int64_t>(256, ceil_div(N, kRoundThreads)));
  auto round = [&](auto kind_c, auto cols_c, auto counts_c, std::atomic<bool> (&flags)[kMaxDevices], const RoundArgs& a) -> int {
    constexpr Gradient kKind = decltype(kind_c)::value;
    constexpr int kCols      = decltype(cols_c)::value;
    constexpr bool kCounts   = decltype(counts_c)::value;
    LBT_TRY((allow_dynamic_lds(round_kernel<kKind, kCols, kCounts>, 3 * kMostSums * sizeof(double), flags)));
    RoundArgs b      = a;
    b.lane_copies    = 1;
    const size_t one = 2 * static_cast<size_t>(a.n_nodes) * K * sizeof(double);
    while (b.lane_copies < kLaneCopies && 2 * b.lane_copies * one <= kCopiesLds) b.lane_copies *= 2;
    const size_t lds = static_cast<size_t>(a.prev_nodes) * K * sizeof(double) + b.lane_copies * one;
    round_kernel<kKind, kCols, kCounts><<<round_grid, kRoundThreads, lds, stream>>>(b);
    return LBT_OK;
  };
  using std::integral_constant;
  using Squared  = integral_constant<Gradient, Gradient::kSquared>;
  using Logistic = integral_constant<Gradient, Gradient::kLogistic>;
  using Softmax  = integral_constant<Gradient, Gradient::kSoftmax>;
  auto run_round = [&](const RoundArgs& a) -> int {
    const std::false_type sums{};
    if (objective == LBT_OBJ_SQUARED_ERROR && weight == nullptr) {
      const std::true_type counts{};
      return K == 1 ? round(Squared{}, integral_constant<int, 1>{}, counts, round_attr[13], a)
                    : round(Squared{}, integral_constant<int, 0>{}, counts, round_attr[14], a);
    }
    if (objective == LBT_OBJ_SQUARED_ERROR)
      return K == 1 ? round(Squared{}, integral_constant<int, 1>{}, sums, round_attr[0], a)
                    : round(Squared{}, integral_constant<int, 0>{}, sums, round_attr[1], a);
    switch (K) {
      case 1: return round(Logistic{}, integral_constant<int, 1>{}, sums, round_attr[2], a);
      case 2: return round(Softmax{}, integral_constant<int, 2>{}, sums, round_attr[3], a);
      case 3: return round(Softmax{}, integral_constant<int, 3>{}, sums, round_attr[4], a);
      case 4: return round(Softmax{}, integral_constant<int, 4>{}, sums, round_attr[5], a);
      case 5: return round(Softmax{}, integral_constant<int, 5>{}, sums, round_attr[6], a);
      case 6: return round(Softmax{}, integral_constant<int, 6>{}, sums, round_attr[7], a);
      case 7: return round(Softmax{}, integral_constant<int, 7>{}, sums, round_attr[8], a);
      case 8: return round(Softmax{}, integral_constant<int, 8>{}, sums, round_attr[9], a);
      case 10: return round(Softmax{}, integral_constant<int, 10>{}, sums, round_attr[10], a);
      case 16: return round(Softmax{}, integral_constant<int, 16>{}, sums, round_attr[11], a);
      default: return round(Softmax{}, integral_constant<int, 0>{}, sums, round_attr[12], a);
    }
  };
  const int slots = static_cast<int>(std::min<int64_t>(n_trees, 2 * p.pass_trees));  // tree t's leaves lie in slot t % slots
  for (int t = 0; t < n_trees;) {
    // trees of this pass: their slots are side by side
    LeavesArgs a{};
    int n = 0, steps = 0;
    while (t + n < n_trees && n < p.pass_trees && (t + n) % slots >= t % slots &&
           static_cast<size_t>(node_off[t + n + 1] - node_off[t]) * sizeof(PackedNode<T>) <= kNodeLds) {
      a.node_off[n] = static_cast<int>(node_off[t + n] - node_off[t]);
      steps         = std::max(steps, depth_of(tree_nodes[t + n]));
      n++;
    }
    a.n_rows     = N;
    a.F          = F;
    a.n_trees    = n;
    a.steps      = steps;
    a.node_words = static_cast<int>((node_off[t + n] - node_off[t]) * sizeof(PackedNode<T>) / 16);
    const bool whole_words = (static_cast<size_t>(F) * sizeof(T)) % 16 == 0;
    a.pitch                = whole_words ? F + 1 : F;
    const size_t node_lds = static_cast<size_t>(a.node_words) * 16, row_bytes = static_cast<size_t>(a.pitch) * sizeof(T);
    a.tile_rows = 256;
    while (a.tile_rows > 64 && node_lds + a.tile_rows * row_bytes > kTwoPerCu) a.tile_rows /= 2;
    const size_t lds  = node_lds + a.tile_rows * row_bytes;
    const bool staged = lds <= kOnePerCu && static_cast<size_t>(F) * sizeof(T) <= static_cast<size_t>(kStagedPerStep) * std::max(steps, 1) * n;
    if (!staged) a.tile_rows = 256;
    a.n_tiles         = ceil_div(N, a.tile_rows);
    uint16_t* to      = row_leaf + static_cast<int64_t>(t % slots) * N;
    const int per_cu  = staged && lds > kTwoPerCu ? 1 : 2;
    const unsigned grid = static_cast<unsigned>(std::min<int64_t>(a.n_tiles, 256 * per_cu));
    // a lane's trees in as few turns as kTogether allows, and as many in each
    const int row_lanes = kLeafThreads / a.tile_rows, trees_each = ceil_div(n, row_lanes);
    const int walks     = ceil_div(trees_each, ceil_div(trees_each, kTogether));
    auto launch         = [&](auto in_lds, auto together) -> int {
      constexpr bool kStaged = decltype(in_lds)::value;
      constexpr int kWalks   = decltype(together)::value;
      static std::atomic<bool> attr[kMaxDevices] = {};
      LBT_TRY((allow_dynamic_lds(tree_leaves_kernel<T, kStaged, kWalks>, kStaged ? kOnePerCu : kNodeLds, attr)));
      tree_leaves_kernel<T, kStaged, kWalks><<<grid, kLeafThreads, kStaged ? lds : node_lds, stream>>>(X, a, nodes + node_off[t], to);
      return LBT_OK;
    };
    auto launch_walks = [&](auto in_lds) -> int {
      switch (walks) {
        case 1: return launch(in_lds, integral_constant<int, 1>{});
        case 2: return launch(in_lds, integral_constant<int, 2>{});
        case 3: return launch(in_lds, integral_constant<int, 3>{});
        default: return launch(in_lds, integral_constant<int, 4>{});
      }
    };
    LBT_TRY((staged ? launch_walks(std::true_type{}) : launch_walks(std::false_type{})));
    for (int end = t + n; t < end; t++) {
      RoundArgs ra{};
      ra.n_rows  = N;
      ra.K       = K;
      ra.n_nodes = tree_nodes[t];
      ra.lr      = lr;
      ra.y       = y;
      ra.weight  = weight;
      ra.pred    = pred;
      ra.leaf    = row_leaf + static_cast<int64_t>(t % slots) * N;
      ra.sums    = sums + sum_off[t];
      if (t > 0) {
        ra.prev_nodes = tree_nodes[t - 1];
        ra.prev_leaf  = row_leaf + static_cast<int64_t>((t - 1) % slots) * N;
        ra.prev_sums  = sums + sum_off[t - 1];
        ra.prev_l1    = l1[t - 1];
        ra.prev_l2    = l2[t - 1];
      }
      LBT_TRY(run_round(ra));
    }
  }
  LBT_TRY(allow_dynamic_lds(finish_trees_kernel, 2 * kMostSums * sizeof(double), finish_attr));
  for (int first = 0; first < n_trees; first += kPackTrees) {
    FinishRefs refs{};
    const int n = std::min(kPackTrees, n_trees - first);
    int widest  = 1;
    for (int i = 0; i < n; i++) {
      refs.feature[i] = feature[first + i];
      refs.sums[i]    = sums + sum_off[first + i];
      refs.leaf[i]    = leaf_out[first + i];
      refs.hessian[i] = hessian_out[first + i];
      refs.l1[i]      = l1[first + i];
      refs.l2[i]      = l2[first + i];
      refs.n_nodes[i] = tree_nodes[first + i];
      widest          = std::max(widest, tree_nodes[first + i]);
    }
    const int adders = first + n == n_trees ? static_cast<int>(std::min<int64_t>(256, ceil_div(N * K, 4096))) : 0;
    finish_trees_kernel<<<n + adders, 1024, 2 * static_cast<size_t>(widest) * K * sizeof(double), stream>>>(
      refs, n, K, row_leaf + static_cast<int64_t>((n_trees - 1) % slots) * N, N * K, pred);
  }
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

}  // namespace
}  // namespace lbt

extern "C" {

size_t lbt_update_trees_workspace_bytes(int64_t n_rows, int32_t n_features, int32_t x_dtype, int32_t n_outputs, int32_t n_trees,
                                        const int32_t* tree_nodes)
{
  if (n_rows < 1 || n_features < 1 || n_outputs < 1 || n_trees < 1 || tree_nodes == nullptr ||
      (x_dtype != LBT_F32 && x_dtype != LBT_F64))
    return 0;
  for (int t = 0; t < n_trees; t++)
    if (tree_nodes[t] < 1) return 0;
  const lbt::Plan p = lbt::make_plan(n_rows, n_features, x_dtype == LBT_F32 ? 4 : 8, n_outputs, n_trees, tree_nodes);
  return p.taken ? p.bytes : 0;
}

int lbt_update_trees(void* stream, const void* X, int32_t x_dtype, int64_t n_rows, int32_t n_features, int32_t objective,
                     const double* y, const double* sample_weight, double learning_rate, int32_t n_outputs, int32_t n_trees,
                     const int32_t* const* feature, const double* const* split, const int32_t* tree_nodes, const double* l1,
                     const double* l2, double* pred, double* const* leaf_out, double* const* hessian_out, void* workspace,
                     size_t workspace_bytes)
{
  LBT_REQUIRE(x_dtype == LBT_F32 || x_dtype == LBT_F64, "unsupported X dtype %d", x_dtype);
  LBT_REQUIRE(objective == LBT_OBJ_SQUARED_ERROR || objective == LBT_OBJ_LOG_LOSS, "unknown objective %d", objective);
  LBT_REQUIRE(n_rows >= 1 && n_features >= 1 && n_outputs >= 1 && n_trees >= 1, "bad shape");
  LBT_REQUIRE(n_rows * n_outputs < (int64_t(1) << 38), "too many elements");
  LBT_REQUIRE(X && y && pred, "null input");
  LBT_REQUIRE(feature && split && tree_nodes && l1 && l2 && leaf_out && hessian_out, "null tree arrays");
  LBT_REQUIRE(pred != y && pred != sample_weight, "pred may not alias the inputs");
  for (int t = 0; t < n_trees; t++)
    LBT_REQUIRE(feature[t] && split[t] && leaf_out[t] && hessian_out[t] && tree_nodes[t] >= 1, "tree %d is incomplete", t);
  const lbt::Plan p = lbt::make_plan(n_rows, n_features, x_dtype == LBT_F32 ? 4 : 8, n_outputs, n_trees, tree_nodes);
  if (!p.taken) {
    lbt::set_error("trees that lbt_update_trees does not take (lbt_update_trees_workspace_bytes is 0): use lbt_update_tree");
    return LBT_ERR_UNSUPPORTED;
  }
  if (!workspace || workspace_bytes < p.bytes) {
    lbt::set_error("workspace missing or too small for lbt_update_trees");
    return LBT_ERR_WORKSPACE;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  lbt::ProfScope ps(LBT_PROF_OTHER, s);
  return x_dtype == LBT_F32
           ? lbt::update_rounds(s, static_cast<const float*>(X), n_rows, n_features, objective, y, sample_weight, learning_rate,
                                n_outputs, n_trees, feature, split, tree_nodes, l1, l2, pred, leaf_out, hessian_out, workspace, p)
           : lbt::update_rounds(s, static_cast<const double*>(X), n_rows, n_features, objective, y, sample_weight, learning_rate,
                                n_outputs, n_trees, feature, split, tree_nodes, l1, l2, pred, leaf_out, hessian_out, workspace, p);
}

}  // extern "C"
