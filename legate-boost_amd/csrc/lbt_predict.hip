// PredictTask and UpdateTreeTask for one MI355X.
//
// Semantics: rapidsai/legate-boost src/models/tree/predict.cu:26-84 (the walk
// and the per-tree, in-order accumulation into a zeroed f64 output) and
// src/models/tree/update_tree.cc:36-122.
#include "lbt_internal.h"
#include "lbt_trees.h"

#include <algorithm>
#include <type_traits>
#include <vector>

namespace lbt {
namespace {

constexpr int kThreads       = 256;
constexpr int kTreesPerLaunch = 96;  // tree descriptors passed by value per launch

struct TreeRef {
  const double* leaf;
  const int32_t* feature;
  const double* split;
  int32_t n_nodes;
  int32_t pad;
};

struct TreeBatch {
  TreeRef t[kTreesPerLaunch];
};

// walk one row through one tree (predict.cu:62-76); the guard on n_nodes keeps
// a malformed tree from reading past its arrays
template <typename T>
__device__ inline int walk(const T* xrow, const TreeRef& tr)
{
  int pos = 0;
  for (int depth = 0; depth < 100; depth++) {
    int ft = tr.feature[pos];
    if (ft == -1) break;
    double xv = static_cast<double>(xrow[ft]);
    int next  = xv <= tr.split[pos] ? 2 * pos + 1 : 2 * pos + 2;
    if (next >= tr.n_nodes) break;
    pos = next;
  }
  return pos;
}

template <typename T, bool kFirst>
__global__ void __launch_bounds__(kThreads)
  predict_kernel(const T* X, int64_t n_rows, int F, TreeBatch batch, int n_trees, int K, const int32_t* wanted,
                 double* out)
{
  if (wanted != nullptr && *wanted == 0) return;
  const int64_t row = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  if (row >= n_rows) return;
  const T* xrow = X + row * F;
  if (K == 1) {
    double acc = kFirst ? 0.0 : out[row];
    for (int t = 0; t < n_trees; t++) acc += batch.t[t].leaf[walk(xrow, batch.t[t])];
    out[row] = acc;
  } else {
    double* o = out + row * K;
    if (kFirst)
      for (int k = 0; k < K; k++) o[k] = 0.0;
    for (int t = 0; t < n_trees; t++) {
      const double* lf = batch.t[t].leaf + static_cast<int64_t>(walk(xrow, batch.t[t])) * K;
      for (int k = 0; k < K; k++) o[k] += lf[k];
    }
  }
}

template <typename T>
int predict_impl(hipStream_t stream, const T* X, int64_t N, int F, int n_trees,
                 const double* const* leaf, const int32_t* const* feature,
                 const double* const* split, const int32_t* tree_nodes, int K, const int32_t* wanted, double* out)
{
  const unsigned grid = static_cast<unsigned>((N + kThreads - 1) / kThreads);
  ProfScope ps(LBT_PROF_PREDICT, stream,
               static_cast<double>(N) * (static_cast<double>(F) * sizeof(T) + K * 8.0));
  int done = 0;
  do {
    TreeBatch b{};
    int n = std::min(kTreesPerLaunch, n_trees - done);
    for (int i = 0; i < n; i++) {
      b.t[i].leaf    = leaf[done + i];
      b.t[i].feature = feature[done + i];
      b.t[i].split   = split[done + i];
      b.t[i].n_nodes = tree_nodes[done + i];
    }
    if (done == 0)
      predict_kernel<T, true><<<grid, kThreads, 0, stream>>>(X, N, F, b, n, K, wanted, out);
    else
      predict_kernel<T, false><<<grid, kThreads, 0, stream>>>(X, N, F, b, n, K, wanted, out);
    done += n;
  } while (done < n_trees);
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

// ---- tiled traversal -------------------------------------------------------
//
// The ensemble is first packed into one array of nodes in the caller's workspace: threshold in
// X's type, feature, and the index of the right child. A leaf is packed as a node that always
// steps to itself (threshold NaN, "right child" = itself), so a walk is a fixed number of
// identical steps with no test for leaves.
// A workgroup then owns a tile of rows (256, or fewer for wide matrices): it stages the rows in
// LDS once and walks them through all trees, a batch of trees at a time that is copied into LDS
// too, so a node step costs two LDS reads and no trip to the L2. Four lanes (8 or 16 for wide
// matrices) share a row and take every fourth tree of the batch, a few trees each, interleaved
// for latency. The nodes of the next batch are
// fetched into registers while the current one is walked, and the leaf values of a batch are
// fetched (from a packed copy) while the next one is walked. They are added in tree order, so a row's sum is formed
// exactly as the per-tree launches of the reference form it.

struct alignas(16) PackedTree {
  int64_t node_off;  // first node in the packed array
  int32_t rel_off;   // and counted from the first node of the tree's batch
  int32_t n_nodes;
};

struct alignas(8) BatchInfo {
  int64_t node_off;  // first node of the batch in the packed array
  int32_t first;     // first tree
  int32_t count;     // trees
  int32_t total;     // nodes
  int32_t steps;     // steps that reach the deepest possible leaf of any tree of the batch
};

// Descriptors are passed by value, 4 KB of arguments a launch; a launch is 3.5 us of the host's time. A prediction of 1000 x 10 with
// 100 trees took 43 us with two of them and a third for the batches, 36 with one (27 with the initial prediction added
// by the kernel for few rows and the stream's handle without an object around it).
constexpr int kPackTrees    = 104; // trees packed per launch
constexpr int kFirstBatches = 10;  // and batch descriptors written by the first one
constexpr int kPackBatches  = 128; // batch descriptors written per launch of their own
constexpr int kTileThreads  = 1024;
// L lanes share a row; a workgroup then covers 1024 / L rows, and a batch holds L * kLaneTrees
// trees. Wide feature matrices take more lanes per row, so that the row tile still fits the LDS.
// kFew: an ensemble of at most L trees (the one tree a boosting round predicts with): one tree
// per lane, so that no lane walks a tree that is not there.
template <int L, bool kFew = false>
struct TileShape {
  static constexpr int kRowLanes   = L;
  static constexpr int kRows       = kTileThreads / L;
  static constexpr int kLaneTrees  = kFew ? 1 : (L == 4 ? 5 : (L == 8 ? 3 : 2));
  static constexpr int kBatchTrees = kRowLanes * kLaneTrees;
};
constexpr size_t kTileLds   = 160 * 1024 - 2048;  // dynamic LDS of the tile kernel
constexpr int kCopyWords    = 6;  // 16-byte words a thread moves per batch: 6 * 1024 * 16 B >= any batch
constexpr int kSmallRunGroups = 256;  // workgroups up to which more lanes share a row: one per CU
constexpr size_t kSmallEnsembleLds = 78 * 1024;  // row tile + nodes of a small ensemble: two workgroups per CU

struct PackBatch {
  const double* leaf[kPackTrees];
  const int32_t* feature[kPackTrees];
  const double* split[kPackTrees];
  int32_t n_nodes[kPackTrees];
  int32_t node_off[kPackTrees];  // from first_node on
  int32_t rel_off[kPackTrees];
  int64_t first_node;
  BatchInfo b[kFirstBatches];
  int32_t first_tree, n_batches;
};
static_assert(sizeof(PackBatch) <= 4096 - 64, "what a launch takes, with the other arguments");
struct BatchTable {
  BatchInfo b[kPackBatches];
};

template <typename T>
__global__ void __launch_bounds__(256)
  pack_trees_kernel(PackBatch b, int F, int K, PackedTree* desc, BatchInfo* batches, PackedNode<T>* nodes, double* leaves)
{
  const int t = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x, n = b.n_nodes[t];
  const int64_t first = b.first_node + b.node_off[t];
  if (t == 0 && i < b.n_batches) batches[i] = b.b[i];
  if (i == 0) {
    PackedTree d;
    d.node_off             = first;
    d.rel_off              = b.rel_off[t];
    d.n_nodes              = n;
    desc[b.first_tree + t] = d;
  }
  if (i < n) nodes[first + i] = pack_node<T>(i, b.feature[t][i], b.split[t][i], F, n);
  // leaf values move along, indexed like the nodes: the workgroup's in one run
  const int64_t from        = static_cast<int64_t>(blockIdx.x) * 256 * K;
  const int here            = min(256, n - static_cast<int>(blockIdx.x) * 256) * K;
  const double* const leaf  = b.leaf[t] + from;
  double* const packed      = leaves + first * K + from;
  for (int e = threadIdx.x; e < here; e += 256) packed[e] = leaf[e];
}

__global__ void write_batches_kernel(BatchTable t, int first, int n, BatchInfo* out)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[first + i] = t.b[i];
}

// The L lanes of a row sit 64 / L lanes apart in their wave: lane = q * (64 / L) + (row of the wave),
// q the row's lane. A quarter wave (what the LDS serves at once) then holds lanes that walk the same
// tree for neighbouring rows: they read neighbouring nodes and, while they agree on the feature,
// neighbouring feature values, where the lanes of one row side by side would read four unrelated trees.
// Lane q of a row owns the trees q * kLaneTrees .. of a batch.
template <int L>
__device__ inline int from_previous_lane_of_row(int v)
{
  // value of the lane 64 / L below (the row's lane q - 1; lane 0 of a row reads its last lane)
  return __shfl(v, (static_cast<int>(threadIdx.x) + 64 - 64 / L) & 63, 64);
}
template <int L>
__device__ inline double from_previous_lane_of_row(double v)
{
  const long long bits = __double_as_longlong(v);
  const int lo = from_previous_lane_of_row<L>(static_cast<int>(bits));
  const int hi = from_previous_lane_of_row<L>(static_cast<int>(bits >> 32));
  return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}
// value of tree jj of a batch, held by lane jj / kLaneTrees of the row's lanes in slot jj % kLaneTrees
template <typename S>
__device__ __forceinline__ int from_owner(const int (&slots)[S::kLaneTrees], int jj)
{
  constexpr int kStride = 64 / S::kRowLanes;
  const int row_in_wave = static_cast<int>(threadIdx.x) & (kStride - 1);
  return __shfl(slots[jj % S::kLaneTrees], (jj / S::kLaneTrees) * kStride + row_in_wave, 64);
}

// What is fetched one batch ahead: the nodes as 16-byte words and where this lane's trees start
// inside the batch.
typedef unsigned int Word16 __attribute__((ext_vector_type(4)));  // plain vector: stays in registers
template <typename S>
struct Prefetched {
  Word16 words[kCopyWords];
  int base[S::kLaneTrees];
};

template <typename T, typename S>
__device__ __forceinline__ Prefetched<S> fetch_batch(const BatchInfo& bi, const PackedNode<T>* __restrict__ nodes,
                                                  const PackedTree* __restrict__ desc, int q)
{
  constexpr int kNodesPerWord = 16 / sizeof(PackedNode<T>);
  Prefetched<S> pf;
  // the packed array is 16-byte aligned and batches start on 16-byte boundaries (see predict_tiled)
  const Word16* src = reinterpret_cast<const Word16*>(nodes + bi.node_off);
  const int n16     = (bi.total + kNodesPerWord - 1) / kNodesPerWord;
#pragma unroll
  for (int c = 0; c < kCopyWords; c++) {
    const int i = threadIdx.x + c * kTileThreads;
    // one tree per lane: words past the batch are not asked for (a single tree is a quarter of
    // one round of the threads); full batches load all of them without a test
    if (S::kLaneTrees > 1 || c * kTileThreads < n16) pf.words[c] = src[i < n16 ? i : 0];
  }
#pragma unroll
  for (int j = 0; j < S::kLaneTrees; j++) {
    const int jj = q * S::kLaneTrees + j;
    pf.base[j]   = desc[bi.first + (jj < bi.count ? jj : 0)].rel_off;  // lanes without a tree walk tree 0 again
  }
  return pf;
}

// Single output: the sum of a row travels along the row's lanes. Lane 0 takes what the last lane
// holds (the sum up to the previous batch), adds the leaf values of its own trees in tree order and
// hands the sum on; after the last lane's turn that lane holds the sum up to this batch. Every lane
// runs every turn (the lanes whose turn it is not keep their value), so the adds of a row happen in
// tree order exactly as the per-tree launches of the reference add them.
template <typename S>
__device__ __forceinline__ void add_in_order(double& run, const double (&val)[S::kLaneTrees], int cnt, int q)
{
#pragma unroll
  for (int turn = 0; turn < S::kRowLanes; turn++) {
    double t = from_previous_lane_of_row<S::kRowLanes>(run);
#pragma unroll
    for (int j = 0; j < S::kLaneTrees; j++) {
      const double a = t + val[j];
      t              = q * S::kLaneTrees + j < cnt ? a : t;
    }
    run = q == turn ? t : run;
  }
}
// Several outputs: the row's lanes share the outputs out, kOwn neighbouring ones each, and every lane adds the
// leaf values of all trees of the batch for its own (in tree order). A tree's leaf of a row is then read once,
// side by side by the row's lanes, eight trees' loads in flight. (With all outputs in every lane each of the
// L lanes fetched the whole leaf again: 500,003 x 200, 50 trees of depth 8 with 8 outputs took 3.89 ms, of
// which the walk is a tenth; now 0.60.) batch_leaves: at this lane's first output; own: how many it has.
template <typename S, int kOwn>
__device__ __forceinline__ void add_leaves_in_order(double (&acc)[kOwn], const int (&at)[S::kLaneTrees], int cnt,
                                                    const double* __restrict__ batch_leaves, int K, int own)
{
  constexpr int kGroup = S::kBatchTrees < 8 ? S::kBatchTrees : 8;
  static_assert(S::kBatchTrees % kGroup == 0 || S::kBatchTrees == 20, "the last group of 20 trees is half full");
#pragma unroll
  for (int first = 0; first < S::kBatchTrees; first += kGroup) {
    if (first < cnt) {
      double v[kGroup][kOwn];
#pragma unroll
      for (int u = 0; u < kGroup; u++) {
        const int jj = first + u;
        if (jj < S::kBatchTrees) {
          const int p      = from_owner<S>(at, jj);
          const double* lf = batch_leaves + static_cast<int64_t>(p) * K;
#pragma unroll
          for (int i = 0; i < kOwn; i++) v[u][i] = jj < cnt && i < own ? lf[i] : 0.0;
        }
      }
#pragma unroll
      for (int u = 0; u < kGroup; u++)
        if (first + u < S::kBatchTrees && first + u < cnt) {
#pragma unroll
          for (int i = 0; i < kOwn; i++) acc[i] += v[u][i];
        }
    }
  }
}

// kOwn: 0 for one output, else the outputs a lane adds up
template <typename T, int kOwn, int L, bool kFew = false>
__global__ void __launch_bounds__(kTileThreads)
  predict_tile_kernel(const T* __restrict__ X, int64_t n_rows, int F, int pitch, int n_batches,
                      const BatchInfo* __restrict__ batches, const PackedTree* __restrict__ desc,
                      const PackedNode<T>* __restrict__ nodes, const double* __restrict__ leaves, int K, int k0,
                      int value_off, const int32_t* __restrict__ wanted, double* __restrict__ out)
{
  // wanted: null, or a device word that is 0 when the rows have been predicted by ranks
  if (wanted != nullptr && *wanted == 0) return;
  // value_off: where the LDS has room for a batch's leaf values (one output, 16 lanes per row), or 0. Handing a row's sum
  // on through 16 lanes is a chain of 16 cross-lane moves per batch; with few rows, when nothing hides it, the
  // values go through the LDS to the first wave instead, a row per lane.
  // k0: first of the (at most L * kOwn) outputs this launch sums; more outputs take a launch per chunk
  constexpr bool kSingle = kOwn == 0;
  using S = TileShape<L, kFew>;
  constexpr int kTileRows = S::kRows, kLaneTrees = S::kLaneTrees;
  extern __shared__ __align__(16) unsigned char smem_raw[];  // 16-byte aligned whatever static LDS precedes it
  T* s_x = reinterpret_cast<T*>(smem_raw);
  const size_t x_bytes = (static_cast<size_t>(kTileRows) * pitch * sizeof(T) + 15) & ~size_t(15);
  PackedNode<T>* s_nodes = reinterpret_cast<PackedNode<T>*>(smem_raw + x_bytes);
  Word16* s_words        = reinterpret_cast<Word16*>(smem_raw + x_bytes);
  constexpr int kNodesPerWord = 16 / sizeof(PackedNode<T>);

  const int64_t row0  = blockIdx.x * static_cast<int64_t>(kTileRows);
  const int rows_here = static_cast<int>(min<int64_t>(kTileRows, n_rows - row0));
  {
    const T* src    = X + row0 * F;
    const int total = rows_here * F;
    if (sizeof(T) == 4 && (F & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0) {
      const float4* src4 = reinterpret_cast<const float4*>(src);
      float* sx          = reinterpret_cast<float*>(s_x);
      for (int i = threadIdx.x; i < total / 4; i += kTileThreads) {
        const float4 v = src4[i];
        const int e = i * 4, r = e / F, f = e - r * F;
        float* d = sx + r * pitch + f;
        d[0] = v.x;
        d[1] = v.y;
        d[2] = v.z;
        d[3] = v.w;
      }
    } else {
      for (int i = threadIdx.x; i < total; i += kTileThreads) {
        const int r = i / F, f = i - r * F;
        s_x[r * pitch + f] = src[i];
      }
    }
  }
  constexpr int kRowsPerWave = 64 / L;
  const int r      = (static_cast<int>(threadIdx.x) >> 6) * kRowsPerWave + (static_cast<int>(threadIdx.x) & (kRowsPerWave - 1));
  const int q      = (static_cast<int>(threadIdx.x) & 63) / kRowsPerWave;
  const bool valid = r < rows_here;
  const T* my_x    = s_x + (valid ? r : 0) * pitch;
  constexpr int kAcc = kSingle ? 1 : kOwn;
  const int k_first  = kSingle ? 0 : k0 + q * kOwn;  // this lane's first output
  double acc[kAcc];
#pragma unroll
  for (int k = 0; k < kAcc; k++) acc[k] = 0.0;

  // fetched one batch ahead: the batch descriptor, the nodes (as 16-byte words) and where this
  // lane's trees start inside the batch
  BatchInfo info_n = batches[0];
  Prefetched<S> pf = fetch_batch<T, S>(info_n, nodes, desc, q);
  double val[kLaneTrees];  // single output: leaf values of this lane's trees of the previous batch
  int cnt_prev = 0;
#pragma unroll
  for (int j = 0; j < kLaneTrees; j++) val[j] = 0.0;

  constexpr bool kValues = kSingle && L == 16 && !kFew;
  double* const s_value  = reinterpret_cast<double*>(smem_raw + value_off);  // [kBatchTrees][kTileRows]
  const bool summing     = kValues && threadIdx.x < 64;
  int handed             = 0;  // trees whose values lie in the LDS
  auto hand_over = [&](int count) {
#pragma unroll
    for (int j = 0; j < kLaneTrees; j++)
      if (q * kLaneTrees + j < count) s_value[(q * kLaneTrees + j) * kTileRows + r] = val[j];
    handed = count;
  };
  auto add_handed = [&]() {
#pragma unroll 8
    for (int jj = 0; jj < handed; jj++) acc[0] += s_value[jj * kTileRows + threadIdx.x];
  };

  for (int b = 0; b < n_batches; b++) {
    const BatchInfo info = info_n;
    __syncthreads();  // the previous batch is no longer read; on the first pass: X tile complete
    {
      const int n16 = (info.total + kNodesPerWord - 1) / kNodesPerWord;
#pragma unroll
      for (int c = 0; c < kCopyWords; c++) {
        const int i = threadIdx.x + c * kTileThreads;
        if (i < n16) s_words[i] = pf.words[c];
      }
    }
    if (summing && value_off != 0) add_handed();
    int base[kLaneTrees], pos[kLaneTrees];
#pragma unroll
    for (int j = 0; j < kLaneTrees; j++) {
      base[j] = pf.base[j];
      pos[j]  = 0;
    }
    __syncthreads();
    if (b + 1 < n_batches) {
      info_n = batches[b + 1];
      pf = fetch_batch<T, S>(info_n, nodes, desc, q);
    }
    for (int s = 0; s < info.steps; s++) {
#pragma unroll
      for (int j = 0; j < kLaneTrees; j++) {
        const PackedNode<T> nd = s_nodes[base[j] + pos[j]];
        if constexpr (sizeof(T) == 4) {
          const float xv = *reinterpret_cast<const float*>(reinterpret_cast<const unsigned char*>(my_x) +
                                                           (nd.feat_right & 0xffffu));
          pos[j]         = static_cast<int>(nd.feat_right >> 16) - (xv <= nd.thr ? 1 : 0);
        } else {
          const double xv = my_x[nd.feat];
          pos[j]          = nd.right - (xv <= nd.thr ? 1 : 0);
        }
      }
    }
    if constexpr (kSingle) {
      // leaf values of the previous batch arrived while this one was walked
      if (kValues && value_off != 0)
        hand_over(cnt_prev);
      else
        add_in_order<S>(acc[0], val, cnt_prev, q);
#pragma unroll
      for (int j = 0; j < kLaneTrees; j++) val[j] = leaves[info.node_off + base[j] + pos[j]];
      cnt_prev = info.count;
    } else {
      int at[kLaneTrees];
#pragma unroll
      for (int j = 0; j < kLaneTrees; j++) at[j] = base[j] + pos[j];
      add_leaves_in_order<S, kAcc>(acc, at, info.count, leaves + info.node_off * K + k_first, K, K - k_first);
    }
  }
  if (kValues && value_off != 0) {
    __syncthreads();
    if (summing) add_handed();
    __syncthreads();
    hand_over(cnt_prev);
    __syncthreads();
    if (summing) add_handed();
    if (summing && static_cast<int>(threadIdx.x) < rows_here) out[row0 + threadIdx.x] = acc[0];
    return;
  }
  if constexpr (kSingle) add_in_order<S>(acc[0], val, cnt_prev, q);
  // single output: the row's last lane holds the sum; several outputs: every lane holds its own
  if (valid && (!kSingle || q == L - 1)) {
    double* o = out + (row0 + r) * K + k_first;
#pragma unroll
    for (int i = 0; i < kAcc; i++)
      if (k_first + i < K) o[i] = acc[i];
  }
}

// ---- few rows
//
// With few rows a call is a chain of latencies: the tile kernel above walks 32 trees at a time, each batch four dependent
// trips to memory and the LDS (256 x 32 with 100 trees of depth 6: 12.3 us). Here a workgroup takes kFewRows rows through
// as many batches at once as the LDS holds, a (row, tree) per lane; everything that is needed first (rows, the nodes from the
// start of the array, the lanes' trees) is asked for before the first wait. The values pass through the LDS to the lanes
// that add a row's in tree order: 7.3 us a launch where the tile kernel takes 12.4 (1000 x 10 f64: 9.9 and 16.7). Ensembles and
// rows that no cache holds, one after the other: 9.8 us a call (the host's time) and 14.3. A workgroup copies the ensemble
// for 16 rows only: with 6433 x 94 and 117 trees of depth 7 it takes 22.0 us and the tile kernel 15.3, with 4096 x 32 and 100
// of depth 6 7.9 and 13.1. An ensemble of at most as many trees as a row has lanes there (up to
// 16) is one batch there too: 52 x 5, 7 trees 3.8 and 3.9 us.
constexpr int kFewRows        = 16;
constexpr int64_t kFewMostRows = 4096;  // one workgroup per CU
constexpr int kFewLanes       = kTileThreads / kFewRows;  // of a row
constexpr int kFewWords       = 8;    // 16-byte words of nodes that a thread moves per turn
constexpr int kFewTogether    = 2;    // trees a lane walks at once
constexpr int kFewGroupTrees  = kFewTogether * kFewLanes;

template <typename T>
__global__ void __launch_bounds__(kTileThreads)
  predict_few_kernel(const T* __restrict__ X, int64_t n_rows, int F, int pitch, int n_trees, int n_batches,
                     const BatchInfo* __restrict__ batches, const PackedTree* __restrict__ desc,
                     const PackedNode<T>* __restrict__ nodes, const double* __restrict__ leaves, int K, int node_at,
                     int cap_words, int cap_trees, int64_t all_words, int value_at, const double* __restrict__ init,
                     double* __restrict__ out)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int kNodesPerWord = 16 / sizeof(PackedNode<T>);
  T* s_x                = reinterpret_cast<T*>(smem_raw);
  PackedNode<T>* s_node = reinterpret_cast<PackedNode<T>*>(smem_raw + node_at);
  double* s_value       = reinterpret_cast<double*>(smem_raw + value_at);  // [tree][row][output]
  const int tid = threadIdx.x, r = tid % kFewRows, q = tid / kFewRows;
  const int64_t row0  = blockIdx.x * static_cast<int64_t>(kFewRows);
  const int rows_here = static_cast<int>(min<int64_t>(kFewRows, n_rows - row0));
  Word16 ahead[kFewWords];
  int64_t tree_at[kFewTogether];
  auto fetch = [&](int64_t first_word, int64_t words) {
    const Word16* src = reinterpret_cast<const Word16*>(nodes) + first_word;
#pragma unroll
    for (int c = 0; c < kFewWords; c++)
      if (tid + c * kTileThreads < words) ahead[c] = src[tid + c * kTileThreads];
  };
  auto fetch_trees = [&](int first) {
#pragma unroll
    for (int j = 0; j < kFewTogether; j++) tree_at[j] = desc[min(first + q + j * kFewLanes, n_trees - 1)].node_off;
  };
  // the first group begins the array; where it ends is not known yet
  fetch(0, min<int64_t>(cap_words, all_words));
  fetch_trees(0);
  for (int i = tid; i < rows_here * F; i += kTileThreads) {
    const int row = i / F;
    s_x[row * pitch + (i - row * F)] = X[row0 * F + i];
  }
  const T* my_x   = s_x + (r < rows_here ? r : 0) * pitch;
  const int items = kFewRows * K;  // (row, output) sums, one a thread
  double acc      = 0.0;
  for (int b = 0; b < n_batches;) {
    // as many batches as fit
    const int64_t start = batches[b].node_off;
    int count = 0, steps = 0;
    int64_t end = start;
    while (b < n_batches) {
      const BatchInfo i = batches[b];
      if ((i.node_off + i.total - start + kNodesPerWord - 1) / kNodesPerWord > cap_words || count + i.count > cap_trees) break;
      end = i.node_off + i.total;
      count += i.count;
      steps = max(steps, i.steps);
      b++;
    }
    if (count == 0) return;  // a batch that does not fit: the host does not launch for such ensembles
    const int words = static_cast<int>((end - start + kNodesPerWord - 1) / kNodesPerWord);
#pragma unroll
    for (int c = 0; c < kFewWords; c++)
      if (tid + c * kTileThreads < words) reinterpret_cast<Word16*>(s_node)[tid + c * kTileThreads] = ahead[c];
    int base[kFewTogether], pos[kFewTogether];
#pragma unroll
    for (int j = 0; j < kFewTogether; j++) {
      base[j] = q + j * kFewLanes < count ? static_cast<int>(tree_at[j] - start) : 0;  // lanes without a tree walk the first again
      pos[j]  = 0;
    }
    __syncthreads();
    if (b < n_batches) {
      const int64_t next = batches[b].node_off / kNodesPerWord;
      fetch(next, min<int64_t>(cap_words, all_words - next));
      fetch_trees(batches[b].first);
    }
    for (int s = 0; s < steps; s++) {
#pragma unroll
      for (int j = 0; j < kFewTogether; j++) pos[j] = step_from<T>(s_node[base[j] + pos[j]], my_x);
    }
#pragma unroll
    for (int j = 0; j < kFewTogether; j++)
      if (q + j * kFewLanes < count) {
        const double* leaf = leaves + (start + base[j] + pos[j]) * K;
        double* value      = s_value + ((q + j * kFewLanes) * kFewRows + r) * K;
        for (int k = 0; k < K; k++) value[k] = leaf[k];
      }
    __syncthreads();
    if (tid < items) {
#pragma unroll 8
      for (int t = 0; t < count; t++) acc += s_value[t * items + tid];
    }
  }
  if (tid < rows_here * K) out[row0 * K + tid] = init != nullptr ? init[tid % K] + acc : acc;
}

// init + the sums, where the kernel that formed them did not add it. kWide: out is 16-byte aligned, two entries at a time
// (300,000 x 8: 10.5 us with one and remainders of 64 bits, which take several times those of 32).
template <bool kWide>
__global__ void __launch_bounds__(kThreads) add_init_kernel(const double* __restrict__ init, int64_t n, int K, double* out)
{
  constexpr int kAtOnce = kWide ? 2 : 1;
  const int64_t i       = kAtOnce * (blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x);
  if (i >= n) return;
  const int k = K == 1 ? 0 : (n >> 32) == 0 ? static_cast<int>(static_cast<uint32_t>(i) % static_cast<uint32_t>(K)) : static_cast<int>(i % K);
  if (kWide && i + 1 < n) {
    double2* const o = reinterpret_cast<double2*>(out + i);
    const double2 v  = *o;
    *o               = make_double2(init[k] + v.x, init[k + 1 == K ? 0 : k + 1] + v.y);
  } else {
    out[i] = init[k] + out[i];
  }
}

size_t padded_nodes(int n_trees, int64_t total_nodes)
{
  return static_cast<size_t>(total_nodes) + 2 * static_cast<size_t>(n_trees);  // batches start on 16 bytes
}
size_t packed_bytes(int n_trees, int64_t total_nodes, int K, size_t node_size)
{
  // tree descriptors, batch descriptors (at most one per tree), nodes, leaf values
  return ((static_cast<size_t>(n_trees) * sizeof(PackedTree) + 255) & ~size_t(255)) +
         ((static_cast<size_t>(n_trees) * sizeof(BatchInfo) + 255) & ~size_t(255)) +
         ((padded_nodes(n_trees, total_nodes) * node_size + 255) & ~size_t(255)) +
         padded_nodes(n_trees, total_nodes) * static_cast<size_t>(K) * sizeof(double) + 512;
}

// Where the parts of a packed ensemble lie in its buffer.
template <typename T>
struct PackedLayout {
  PackedTree* desc;
  BatchInfo* batches;
  PackedNode<T>* nodes;
  double* leaves;
  PackedLayout(void* buffer, int n_trees, int64_t total_nodes)
  {
    const size_t desc_bytes  = (static_cast<size_t>(n_trees) * sizeof(PackedTree) + 255) & ~size_t(255);
    const size_t batch_bytes = (static_cast<size_t>(n_trees) * sizeof(BatchInfo) + 255) & ~size_t(255);
    const size_t node_bytes  = (padded_nodes(n_trees, total_nodes) * sizeof(PackedNode<T>) + 255) & ~size_t(255);
    uintptr_t raw            = (reinterpret_cast<uintptr_t>(buffer) + 255) & ~uintptr_t(255);
    desc                     = reinterpret_cast<PackedTree*>(raw);
    batches                  = reinterpret_cast<BatchInfo*>(raw + desc_bytes);
    nodes                    = reinterpret_cast<PackedNode<T>*>(raw + desc_bytes + batch_bytes);
    leaves                   = reinterpret_cast<double*>(raw + desc_bytes + batch_bytes + node_bytes);
  }
};

// Lanes per row of the tile kernel for rows of F values: as few as keep the row tile within
// about half of the LDS; 0 when no shape fits.
template <typename T>
int tile_lanes(int F, size_t* x_bytes)
{
  const int pitch = F | 1;  // odd pitch: the rows of a wave start in different LDS banks
  for (int l : {4, 8, 16}) {
    *x_bytes = (static_cast<size_t>(kTileThreads / l) * pitch * sizeof(T) + 15) & ~size_t(15);
    if (*x_bytes <= kTileLds * 55 / 100) return l;
  }
  return 0;
}

// Packs the trees for the tile kernel into `buffer`. Returns LBT_OK and fills *ens when the
// shapes fit the tile kernel; leaves ens->data null when they do not.
template <typename T>
int pack_tiled(hipStream_t stream, int F, int n_trees, const double* const* leaf, const int32_t* const* feature,
               const double* const* split, const int32_t* tree_nodes, int K, void* buffer, size_t buffer_bytes,
               lbt_packed_ensemble* ens)
{
  *ens = lbt_packed_ensemble{};
  if (buffer == nullptr || F > kMaxPackedFeatures) return LBT_OK;
  int64_t total_nodes = 0;
  int max_nodes       = 0;
  for (int i = 0; i < n_trees; i++) {
    total_nodes += tree_nodes[i];
    max_nodes = std::max(max_nodes, tree_nodes[i]);
  }
  size_t x_bytes = 0;
  int lanes      = tile_lanes<T>(F, &x_bytes);
  if (lanes == 0) return LBT_OK;
  // A small ensemble spends its time streaming X: then a narrower row tile that lets two
  // workgroups share a CU (one loads while the other walks) beats the widest tile that fits.
  const size_t all_nodes = static_cast<size_t>(total_nodes + 2 * n_trees) * sizeof(PackedNode<T>);
  if (all_nodes <= 24 * 1024) {
    for (int l : {4, 8, 16}) {
      const size_t xb = (static_cast<size_t>(kTileThreads / l) * (F | 1) * sizeof(T) + 15) & ~size_t(15);
      if (l >= lanes && xb + all_nodes <= kSmallEnsembleLds) {
        lanes   = l;
        x_bytes = xb;
        break;
      }
    }
  }
  const bool few        = n_trees <= lanes;
  const int batch_trees = few ? lanes
                              : (lanes == 4 ? TileShape<4>::kBatchTrees
                                            : (lanes == 8 ? TileShape<8>::kBatchTrees : TileShape<16>::kBatchTrees));
  constexpr int kNodesPerWord = 16 / sizeof(PackedNode<T>);
  const int64_t node_cap = std::min<int64_t>(static_cast<int64_t>((kTileLds - x_bytes) / sizeof(PackedNode<T>)),
                                             static_cast<int64_t>(kCopyWords) * kTileThreads * kNodesPerWord);
  if (max_nodes > node_cap || max_nodes > kMaxPackedNodes) return LBT_OK;
  const size_t need = packed_bytes(n_trees, total_nodes, K, sizeof(PackedNode<T>));
  if (buffer_bytes < need) {
    set_error("packed ensemble buffer too small: %zu bytes given, %zu needed", buffer_bytes, need);
    return LBT_ERR_WORKSPACE;
  }
  PackedLayout<T> lay(buffer, n_trees, total_nodes);

  // batches: consecutive trees, at most batch_trees, whose nodes fit the LDS share together
  std::vector<BatchInfo> binfo;
  std::vector<int64_t> node_off(n_trees);
  std::vector<int32_t> rel_off(n_trees);
  int64_t off = 0, widest_batch = 0;
  for (int t = 0; t < n_trees;) {
    off = (off + kNodesPerWord - 1) / kNodesPerWord * kNodesPerWord;  // 16-byte aligned start
    BatchInfo bi{};
    bi.node_off = off;
    bi.first    = t;
    int64_t in_batch = 0;
    while (t < n_trees && bi.count < batch_trees && in_batch + tree_nodes[t] <= node_cap) {
      node_off[t] = off + in_batch;
      rel_off[t]  = static_cast<int32_t>(in_batch);
      int steps   = 0;
      while (((int64_t(1) << (steps + 1)) - 1) < tree_nodes[t]) steps++;
      bi.steps = std::max(bi.steps, steps);
      in_batch += tree_nodes[t];
      bi.count++;
      t++;
    }
    bi.total = static_cast<int32_t>(in_batch);
    off += in_batch;
    widest_batch = std::max(widest_batch, in_batch);
    binfo.push_back(bi);
  }
  const int n_batches = static_cast<int>(binfo.size());
  for (int first = 0; first < n_trees; first += kPackTrees) {
    PackBatch b;
    const int n = std::min(kPackTrees, n_trees - first);
    int widest  = 1;
    b.first_node = node_off[first];
    b.first_tree = first;
    b.n_batches  = first == 0 ? std::min(n_batches, kFirstBatches) : 0;
    for (int i = 0; i < b.n_batches; i++) b.b[i] = binfo[i];
    for (int i = 0; i < n; i++) {
      b.leaf[i]     = leaf[first + i];
      b.feature[i]  = feature[first + i];
      b.split[i]    = split[first + i];
      b.n_nodes[i]  = tree_nodes[first + i];
      b.node_off[i] = static_cast<int32_t>(node_off[first + i] - b.first_node);
      b.rel_off[i]  = rel_off[first + i];
      widest        = std::max(widest, tree_nodes[first + i]);
    }
    dim3 grid(static_cast<unsigned>((widest + 255) / 256), n);
    pack_trees_kernel<T><<<grid, 256, 0, stream>>>(b, F, K, lay.desc, lay.batches, lay.nodes, lay.leaves);
  }
  for (int first = kFirstBatches; first < n_batches; first += kPackBatches) {
    BatchTable tb{};
    const int n = std::min(kPackBatches, n_batches - first);
    for (int i = 0; i < n; i++) tb.b[i] = binfo[first + i];
    write_batches_kernel<<<1, kPackBatches, 0, stream>>>(tb, first, n, lay.batches);
  }
  LBT_HIP(hipGetLastError());
  ens->data        = buffer;
  ens->bytes       = buffer_bytes;
  ens->x_dtype     = sizeof(T) == 4 ? LBT_F32 : LBT_F64;
  ens->n_features  = F;
  ens->n_outputs   = K;
  ens->n_trees     = n_trees;
  ens->n_batches   = n_batches;
  ens->lanes       = lanes;
  ens->few_trees   = few ? 1 : 0;
  // the row tile and the widest batch of nodes (whole 16-byte words)
  ens->lds_bytes   = static_cast<int32_t>(
    x_bytes + ((static_cast<size_t>(widest_batch + kNodesPerWord) * sizeof(PackedNode<T>) + 15) & ~size_t(15)));
  ens->total_nodes = total_nodes;
  return LBT_OK;
}

// Whether the tile kernel with 16 lanes per row has room for the values of a batch beside rows and nodes.
constexpr size_t kBatchValues = static_cast<size_t>(TileShape<16>::kBatchTrees) * TileShape<16>::kRows * sizeof(double);
size_t values_offset(const lbt_packed_ensemble& ens) { return (static_cast<size_t>(ens.lds_bytes) + 15) & ~size_t(15); }
bool values_through_lds(const lbt_packed_ensemble& ens) { return ens.n_outputs == 1 && values_offset(ens) + kBatchValues <= kTileLds; }

// *init (optional): what the sums are added to; null afterwards where that has been done.
// The kernel for few rows over a packed ensemble; *done stays false where the tile kernel is the faster one or the shapes
// do not fit.
template <typename T>
int run_few(hipStream_t stream, const T* X, int64_t N, const lbt_packed_ensemble& ens, const double** init, double* out, bool* done)
{
  const int F = ens.n_features, K = ens.n_outputs, pitch = F | 1;
  if (ens.few_trees != 0 || N > kFewMostRows || kFewRows * K > kTileThreads) return LBT_OK;
  constexpr int kNodesPerWord = 16 / sizeof(PackedNode<T>);
  const size_t x_bytes     = (static_cast<size_t>(kFewRows) * pitch * sizeof(T) + 15) & ~size_t(15);
  const size_t tree_values = static_cast<size_t>(kFewRows) * K * sizeof(double);
  // a batch holds at most 32 trees; the rest of the values' share is for more of them
  const int cap_trees = static_cast<int>(std::max<size_t>(32, std::min<size_t>(std::min(kFewGroupTrees, ens.n_trees), 32 * 1024 / tree_values)));
  const size_t value_bytes = cap_trees * tree_values;
  if (x_bytes + value_bytes >= kTileLds) return LBT_OK;
  const int64_t all_words = (ens.total_nodes + ens.n_batches + kNodesPerWord - 1) / kNodesPerWord;  // batches start on whole words
  const int64_t room      = static_cast<int64_t>((kTileLds - x_bytes - value_bytes) / 16);
  const int64_t cap_words = std::min<int64_t>({room, all_words, static_cast<int64_t>(kFewWords) * kTileThreads});
  const size_t tile_rows  = kTileThreads / ens.lanes;
  const size_t tile_x     = (tile_rows * pitch * sizeof(T) + 15) & ~size_t(15);  // lds_bytes: that and the widest batch
  const int64_t widest    = static_cast<int64_t>(static_cast<size_t>(ens.lds_bytes) - tile_x) / 16 - 1;
  if (widest > cap_words && cap_words < all_words) return LBT_OK;
  // Turns of one batch (of deep trees): most lanes have no tree, and a workgroup copies the ensemble for 16 rows where one of the
  // tile kernel with 16 lanes per row does for 64. Where that one passes values through the LDS as well it is the faster one, and
  // with several outputs below eight trees a batch. Tile kernel and this one, 256 rows, us: 1000 trees of depth 8 on
  // 32 features 124.8 : 163.9, on 10 f64 284 : 322, 300 of depth 8 38.9 : 46.3, 100 of depth 10 45.3 : 56.3; 88 of depth 9
  // on 15 f64 with 8 outputs 56.9 : 66.4. Without values through the LDS: 1000 of depth 8 on 160 features 196 : 170, 300 of
  // depth 8 on 32 f64 130 : 104, with 3 outputs and 20 trees a batch 72.4 : 46.5. Two batches a turn: 300 of depth 7 on 100
  // features 31.3 : 22.4.
  const bool one_batch = 2 * widest > cap_words && cap_words < all_words;
  if (one_batch && (values_through_lds(ens) || (K > 1 && ens.n_trees < 8 * ens.n_batches))) return LBT_OK;
  PackedLayout<T> lay(ens.data, ens.n_trees, ens.total_nodes);
  const int node_at  = static_cast<int>(x_bytes);
  const int value_at = static_cast<int>(x_bytes + cap_words * 16);
  ProfScope ps(LBT_PROF_PREDICT, stream, static_cast<double>(N) * (static_cast<double>(F) * sizeof(T) + K * 8.0));
  static std::atomic<bool> attr[kMaxDevices] = {};
  LBT_TRY(allow_dynamic_lds(predict_few_kernel<T>, kTileLds, attr));
  predict_few_kernel<T><<<static_cast<unsigned>((N + kFewRows - 1) / kFewRows), kTileThreads, value_at + value_bytes, stream>>>(
    X, N, F, pitch, ens.n_trees, ens.n_batches, lay.batches, lay.desc, lay.nodes, lay.leaves, K, node_at,
    static_cast<int>(cap_words), cap_trees, all_words, value_at, init != nullptr ? *init : nullptr, out);
  LBT_HIP(hipGetLastError());
  if (init != nullptr) *init = nullptr;
  *done = true;
  return LBT_OK;
}

// The tile kernel over a packed ensemble.
template <typename T>
int run_tiled(hipStream_t stream, const T* X, int64_t N, const lbt_packed_ensemble& ens, double* out,
              const int32_t* wanted = nullptr, const double** init = nullptr)
{
  const int F = ens.n_features, K = ens.n_outputs, n_batches = ens.n_batches;
  if (wanted == nullptr) {
    bool done = false;
    LBT_TRY(run_few<T>(stream, X, N, ens, init, out, &done));
    if (done) return LBT_OK;
  }
  // The lanes the ensemble was laid out for suit many rows. Batches of so many trees fit the kernels for more lanes
  // per row too (their last lanes then have no tree), and where the rows would leave most CUs without a
  // workgroup these split them further and walk fewer trees per lane: 256 x 32, 100 trees of depth 6: 19.0 us
  // with 4 lanes (one workgroup), 12.3 with 16 and the values through the LDS (18.7 with the sum handed on).
  int lanes = ens.lanes;
  for (const int more : {8, 16})
    if (more > lanes && N <= static_cast<int64_t>(kTileThreads / more) * kSmallRunGroups) lanes = more;
  PackedLayout<T> lay(ens.data, ens.n_trees, ens.total_nodes);
  const int pitch     = F | 1;
  const int tile_rows = kTileThreads / lanes;
  ProfScope ps(LBT_PROF_PREDICT, stream, static_cast<double>(N) * (static_cast<double>(F) * sizeof(T) + K * 8.0));
  const unsigned tiles = static_cast<unsigned>((N + tile_rows - 1) / tile_rows);
  // A walk sums up to one output per lane of a row, or two where there are more; the rest is walked chunk by
  // chunk (each chunk's sums are formed in tree order, as in one walk).
  const int own   = K == 1 ? 0 : (K <= lanes ? 1 : 2);
  const int chunk = K == 1 ? 1 : lanes * own;
  const bool by_values = lanes == 16 && tiles <= kSmallRunGroups && values_through_lds(ens);
  const int value_off  = by_values ? static_cast<int>(values_offset(ens)) : 0;
  const size_t lds     = by_values ? values_offset(ens) + kBatchValues : static_cast<size_t>(ens.lds_bytes);
  auto launch = [&](auto kernel, std::atomic<bool> (&flags)[kMaxDevices]) -> int {
    LBT_TRY(allow_dynamic_lds(kernel, kTileLds, flags));
    for (int k0 = 0; k0 < K; k0 += chunk)
      kernel<<<tiles, kTileThreads, lds, stream>>>(X, N, F, pitch, n_batches, lay.batches, lay.desc, lay.nodes, lay.leaves,
                                                   K, k0, value_off, wanted, out);
    return LBT_OK;
  };
  static std::atomic<bool> attr[2][3][3][kMaxDevices] = {};
  auto shaped = [&](auto lanes_c, auto own_c) -> int {
    constexpr int kL = decltype(lanes_c)::value, kO = decltype(own_c)::value;
    constexpr int at = kL == 4 ? 0 : (kL == 8 ? 1 : 2);
    return ens.few_trees == 1 ? launch(predict_tile_kernel<T, kO, kL, true>, attr[1][at][kO])
                              : launch(predict_tile_kernel<T, kO, kL>, attr[0][at][kO]);
  };
  auto with_lanes = [&](auto lanes_c) -> int {
    if (own == 0) return shaped(lanes_c, std::integral_constant<int, 0>{});
    if (own == 1) return shaped(lanes_c, std::integral_constant<int, 1>{});
    return shaped(lanes_c, std::integral_constant<int, 2>{});
  };
  if (lanes == 4)
    LBT_TRY(with_lanes(std::integral_constant<int, 4>{}));
  else if (lanes == 8)
    LBT_TRY(with_lanes(std::integral_constant<int, 8>{}));
  else
    LBT_TRY(with_lanes(std::integral_constant<int, 16>{}));
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

// Returns LBT_OK and sets *done when the tiled path ran; leaves *done false when the shapes
// do not fit it (then the caller takes the per-node path).
template <typename T>
int predict_tiled(hipStream_t stream, const T* X, int64_t N, int F, int n_trees, const double* const* leaf,
                  const int32_t* const* feature, const double* const* split, const int32_t* tree_nodes, int K,
                  const int32_t* wanted, const double** init, double* out, void* workspace, size_t workspace_bytes, bool* done)
{
  *done = false;
  lbt_packed_ensemble ens;
  LBT_TRY(pack_tiled<T>(stream, F, n_trees, leaf, feature, split, tree_nodes, K, workspace, workspace_bytes, &ens));
  if (ens.data == nullptr) return LBT_OK;
  LBT_TRY(run_tiled<T>(stream, X, N, ens, out, wanted, init));
  *done = true;
  return LBT_OK;
}

// By ranks where that is the faster way and the workspace has the room, else tiled, else per node.
template <typename T>
int predict_any(hipStream_t stream, const T* X, int64_t N, int F, int n_trees, const double* const* leaf,
                const int32_t* const* feature, const double* const* split, const int32_t* tree_nodes, int K, const double** init,
                double* out, void* workspace, size_t workspace_bytes)
{
  int64_t total = 0;
  for (int i = 0; i < n_trees; i++) total += tree_nodes[i];
  const size_t packed = (packed_bytes(n_trees, total, K, sizeof(PackedNode<T>)) + 255) & ~size_t(255);
  const int32_t* wanted = nullptr;
  bool done = false;
  if (workspace != nullptr && workspace_bytes > packed) {
    LBT_TRY(predict_ranked<T>(stream, X, N, F, n_trees, leaf, feature, split, tree_nodes, K, out,
                              static_cast<char*>(workspace) + packed, workspace_bytes - packed, &done, &wanted));
    // wanted: only the device knows whether the ranks sufficed; what follows then runs or ends at once (0.14 ms of a call with
    // 1000 trees of depth 8 for packing and a launch that reads one word)
    if (done && wanted == nullptr) return LBT_OK;
  }
  LBT_TRY(predict_tiled<T>(stream, X, N, F, n_trees, leaf, feature, split, tree_nodes, K, wanted, init, out, workspace,
                           workspace_bytes, &done));
  if (done) return LBT_OK;
  return predict_impl<T>(stream, X, N, F, n_trees, leaf, feature, split, tree_nodes, K, wanted, out);
}

// ---- update

__global__ void zero_doubles_kernel(double* a, int64_t n)
{
  int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (i < n) a[i] = 0.0;
}

// Every node on a row's path receives the row's (g, h) (update_tree.cc:76-90). The sums of an
// inner node are the sums of its children, so a row adds to the node it stops in only and
// finish_update_kernel fills in the rest. A workgroup collects its rows in an LDS copy of the
// node sums (when that fits) and adds the copy to the global sums once; the tree lies in the LDS too.
// What bounds it is how X is read. Walking it in place asks for a cache line per step and row, and the lines of the
// rows in flight do not stay in the L2 (1,000,000 x 50, depth 8: 111 us, the rate of about eight million
// scattered lines), so rows of up to kStagedBytesPerStep bytes per step of the walk are read whole, side by side,
// into the LDS first (59 us). row_leaf, if given, receives the node every row stops in.
constexpr int kUpdateThreads      = 1024;
constexpr int kUpdateLdsDoubles   = 8192;  // node sums up to 64 KB
constexpr int kStagedThreads      = 512;  // tiles of wide rows have fewer of them, but all threads stage (256: 75 us a tree where 512 take 67)
constexpr int kStagedBytesPerStep = 80;    // a scattered line costs as much as about 100 bytes in sequence
constexpr size_t kStagedTile      = 60 * 1024;
enum class UpdateMode { kGlobal, kLds, kStaged };  // where sums and tree lie; kStaged: rows in the LDS too

struct UpdateArgs {
  int64_t n_rows;
  int F, K, n_nodes;
  const double* g;
  const double* h;
  const int32_t* feature;
  const double* split;
  double* G;  // [n_nodes][K]
  double* H;
  int32_t* row_leaf;
  int tile_rows;  // kStaged: a multiple of 64, at most kStagedThreads
  int pitch;      // odd: the rows of a wave start in different banks
};

__host__ __device__ inline size_t update_lds_bytes(int n_nodes, int K)
{
  return (static_cast<size_t>(n_nodes) * (2 * K * sizeof(double) + sizeof(double) + sizeof(int32_t)) + 15) & ~size_t(15);
}

template <typename T, UpdateMode kMode>
__global__ void __launch_bounds__(kUpdateThreads) update_accumulate_kernel(const T* __restrict__ X, UpdateArgs a)
{
  constexpr bool kUseLds = kMode != UpdateMode::kGlobal;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double* s_sum   = reinterpret_cast<double*>(smem_raw);  // [2][K][n_nodes]: nodes side by side in the banks
  double* s_split = s_sum + 2 * static_cast<size_t>(a.n_nodes) * a.K;
  int32_t* s_feat = reinterpret_cast<int32_t*>(s_split + a.n_nodes);
  const int n_sums = a.n_nodes * a.K, tid = threadIdx.x, threads = blockDim.x;
  if constexpr (kUseLds) {
    for (int i = tid; i < 2 * n_sums; i += threads) s_sum[i] = 0.0;
    for (int i = tid; i < a.n_nodes; i += threads) {
      s_split[i] = a.split[i];
      s_feat[i]  = a.feature[i];
    }
    __syncthreads();
  }
  auto take = [&](const T* xrow, int64_t row) {
    int pos = 0;
    for (int depth = 0; depth < 100; depth++) {
      const int ft = kUseLds ? s_feat[pos] : a.feature[pos];
      if (ft == -1) break;
      const double xv = static_cast<double>(xrow[ft]);
      const int next  = xv <= (kUseLds ? s_split[pos] : a.split[pos]) ? 2 * pos + 1 : 2 * pos + 2;
      if (next >= a.n_nodes) break;
      pos = next;
    }
    if (a.row_leaf != nullptr) a.row_leaf[row] = pos;
    for (int k = 0; k < a.K; k++) {
      const double gv = a.g[row * a.K + k], hv = a.h[row * a.K + k];
      if constexpr (kUseLds) {
        unsafeAtomicAdd(&s_sum[k * a.n_nodes + pos], gv);
        unsafeAtomicAdd(&s_sum[n_sums + k * a.n_nodes + pos], hv);
      } else {
        unsafeAtomicAdd(&a.G[static_cast<int64_t>(pos) * a.K + k], gv);
        unsafeAtomicAdd(&a.H[static_cast<int64_t>(pos) * a.K + k], hv);
      }
    }
  };
  if constexpr (kMode == UpdateMode::kStaged) {
    T* s_x = reinterpret_cast<T*>(smem_raw + update_lds_bytes(a.n_nodes, a.K));  // [tile_rows][pitch]
    const int64_t tiles = (a.n_rows + a.tile_rows - 1) / a.tile_rows;
    const bool wide     = sizeof(T) == 4 && (a.F & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0;
    for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
      const int64_t row0 = tile * a.tile_rows;
      const int here     = static_cast<int>(min<int64_t>(a.tile_rows, a.n_rows - row0));
      const T* src       = X + row0 * a.F;
      const int total    = here * a.F;
      __syncthreads();  // the tile before is no longer read
      if (wide) {
        const float4* src4 = reinterpret_cast<const float4*>(src);
#pragma unroll 4
        for (int i = tid; i < total / 4; i += kStagedThreads) {
          const float4 v = src4[i];
          const int r    = i / (a.F / 4);
          T* d           = s_x + r * a.pitch + (i - r * (a.F / 4)) * 4;
          d[0] = v.x;
          d[1] = v.y;
          d[2] = v.z;
          d[3] = v.w;
        }
      } else {
#pragma unroll 4
        for (int i = tid; i < total; i += kStagedThreads) {
          const int r = i / a.F;
          s_x[r * a.pitch + (i - r * a.F)] = src[i];
        }
      }
      __syncthreads();
      if (tid < here) take(s_x + tid * a.pitch, row0 + tid);
    }
  } else {
    for (int64_t row = blockIdx.x * static_cast<int64_t>(threads) + tid; row < a.n_rows;
         row += static_cast<int64_t>(gridDim.x) * threads)
      take(X + row * a.F, row);
  }
  if constexpr (kUseLds) {
    __syncthreads();
    for (int i = tid; i < n_sums; i += threads) {
      const int node = i / a.K, at = (i - node * a.K) * a.n_nodes + node;
      const double gv = s_sum[at], hv = s_sum[n_sums + at];
      if (gv != 0.0) unsafeAtomicAdd(&a.G[i], gv);
      if (hv != 0.0) unsafeAtomicAdd(&a.H[i], hv);
    }
  }
}

// Sums of inner nodes, deepest level first: a node that leads on (the walk above leaves it)
// adds what its two children hold. One workgroup. kUseLds: in the LDS, where a level costs no trip to the L2, and
// with the leaf values (update_tree.cc:104-117) at the end.
template <bool kUseLds>
__global__ void __launch_bounds__(1024)
  finish_update_kernel(const int32_t* __restrict__ feature, int n_nodes, int K, double* G, double* H, double l1, double l2,
                       double* leaf_out, double* hessian_out)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int64_t n = static_cast<int64_t>(n_nodes) * K;
  double* const g = kUseLds ? reinterpret_cast<double*>(smem_raw) : G;
  double* const h = kUseLds ? g + n : H;
  if constexpr (kUseLds) {
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
      g[i] = G[i];
      h[i] = H[i];
    }
    __syncthreads();
  }
  sum_inner_nodes(feature, n_nodes, K, g, h);
  if constexpr (kUseLds) {
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
      const double hv = h[i];
      leaf_out[i]     = updated_leaf(g[i], hv, l1, l2);
      hessian_out[i]  = hv;
    }
  }
}

// update_tree.cc:104-117, for trees whose sums do not fit the LDS
__global__ void update_leaves_kernel(const double* G, const double* H, int64_t n, double l1, double l2,
                                     double* leaf_out, double* hessian_out)
{
  int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (i < n) {
    double hv      = H[i];
    leaf_out[i]    = updated_leaf(G[i], hv, l1, l2);
    hessian_out[i] = hv;
  }
}

template <typename T>
int update_impl(hipStream_t stream, const T* X, UpdateArgs a, double l1, double l2, double* leaf_out,
                double* hessian_out)
{
  const int64_t n = static_cast<int64_t>(a.n_nodes) * a.K;
  zero_doubles_kernel<<<static_cast<unsigned>((2 * n + 255) / 256), 256, 0, stream>>>(a.G, 2 * n);
  const bool lds = 2 * n <= kUpdateLdsDoubles;
  int depth = 0;
  while (((int64_t(1) << (depth + 1)) - 1) < a.n_nodes) depth++;
  const size_t row_bytes = static_cast<size_t>(a.F | 1) * sizeof(T);
  a.pitch                = a.F | 1;
  a.tile_rows            = static_cast<int>(std::min<size_t>(kStagedThreads, kStagedTile / row_bytes / 64 * 64));
  const size_t tree_lds  = update_lds_bytes(a.n_nodes, a.K);
  const size_t lds_bytes = tree_lds + a.tile_rows * row_bytes;
  if (a.n_rows > 0) {
    static std::atomic<bool> attr[2][kMaxDevices] = {};
    const int64_t per_launch = (a.n_rows + kUpdateThreads - 1) / kUpdateThreads;
    const unsigned grid      = static_cast<unsigned>(std::min<int64_t>(per_launch, 512));
    if (lds && a.tile_rows > 0 && static_cast<size_t>(a.F) * sizeof(T) <= static_cast<size_t>(kStagedBytesPerStep) * depth &&
        lds_bytes <= kTileLds) {
      const int per_cu         = std::max(1, static_cast<int>(kTileLds / lds_bytes));
      const int64_t tiles      = (a.n_rows + a.tile_rows - 1) / a.tile_rows;
      const unsigned tile_grid = static_cast<unsigned>(std::min<int64_t>(tiles, 256 * std::min(per_cu, 4)));
      LBT_TRY((allow_dynamic_lds(update_accumulate_kernel<T, UpdateMode::kStaged>, kTileLds, attr[0])));
      update_accumulate_kernel<T, UpdateMode::kStaged><<<tile_grid, kStagedThreads, lds_bytes, stream>>>(X, a);
    } else if (lds) {
      LBT_TRY((allow_dynamic_lds(update_accumulate_kernel<T, UpdateMode::kLds>, 128 * 1024, attr[1])));
      update_accumulate_kernel<T, UpdateMode::kLds><<<grid, kUpdateThreads, tree_lds, stream>>>(X, a);
    } else {
      update_accumulate_kernel<T, UpdateMode::kGlobal><<<grid, kUpdateThreads, 0, stream>>>(X, a);
    }
  }
  if (lds) {
    static std::atomic<bool> attr[kMaxDevices] = {};
    LBT_TRY(allow_dynamic_lds(finish_update_kernel<true>, kUpdateLdsDoubles * sizeof(double), attr));
    finish_update_kernel<true><<<1, 1024, 2 * n * sizeof(double), stream>>>(a.feature, a.n_nodes, a.K, a.G, a.H, l1, l2,
                                                                           leaf_out, hessian_out);
  } else {
    finish_update_kernel<false><<<1, 1024, 0, stream>>>(a.feature, a.n_nodes, a.K, a.G, a.H, l1, l2, leaf_out, hessian_out);
    update_leaves_kernel<<<static_cast<unsigned>((n + 255) / 256), 256, 0, stream>>>(a.G, a.H, n, l1, l2, leaf_out,
                                                                                     hessian_out);
  }
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

}  // namespace
}  // namespace lbt

extern "C" {

int lbt_predict_from(void* stream, const void* X, int32_t x_dtype, int64_t n_rows, int32_t n_features,
                     int32_t n_trees, const double* const* leaf, const int32_t* const* feature,
                     const double* const* split, const int32_t* tree_nodes, int32_t n_outputs,
                     const double* init, double* out, void* workspace, size_t workspace_bytes)
{
  LBT_REQUIRE(x_dtype == LBT_F32 || x_dtype == LBT_F64, "unsupported X dtype %d", x_dtype);
  LBT_REQUIRE(n_features >= 1 && n_outputs >= 1 && n_trees >= 0, "bad shape");
  // predict.cu:35: a shard without rows has nothing to do
  if (n_rows < 1) return LBT_OK;
  LBT_REQUIRE(X && out, "null X or output");
  const int64_t n = n_rows * n_outputs;
  LBT_REQUIRE(init == nullptr || reinterpret_cast<uintptr_t>(init + n_outputs) <= reinterpret_cast<uintptr_t>(out) ||
                reinterpret_cast<uintptr_t>(out + n) <= reinterpret_cast<uintptr_t>(init),
              "the initial prediction and the output overlap");
  LBT_REQUIRE(n_trees == 0 || (leaf && feature && split && tree_nodes), "null tree arrays");
  for (int i = 0; i < n_trees; i++)
    LBT_REQUIRE(leaf[i] && feature[i] && split[i] && tree_nodes[i] >= 1, "tree %d is incomplete", i);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (n_trees == 0) {
    lbt::zero_doubles_kernel<<<static_cast<unsigned>((n + 255) / 256), 256, 0, s>>>(out, n);
  } else if (x_dtype == LBT_F32) {
    LBT_TRY(lbt::predict_any<float>(s, static_cast<const float*>(X), n_rows, n_features, n_trees, leaf, feature, split,
                                    tree_nodes, n_outputs, &init, out, workspace, workspace_bytes));
  } else {
    LBT_TRY(lbt::predict_any<double>(s, static_cast<const double*>(X), n_rows, n_features, n_trees, leaf, feature, split,
                                     tree_nodes, n_outputs, &init, out, workspace, workspace_bytes));
  }
  if (init != nullptr) {
    lbt::ProfScope ps(LBT_PROF_OTHER, s, static_cast<double>(n) * 16.0);
    const bool wide     = reinterpret_cast<uintptr_t>(out) % 16 == 0;
    const int64_t per   = (wide ? 2 : 1) * lbt::kThreads;
    const unsigned grid = static_cast<unsigned>((n + per - 1) / per);
    if (wide)
      lbt::add_init_kernel<true><<<grid, lbt::kThreads, 0, s>>>(init, n, n_outputs, out);
    else
      lbt::add_init_kernel<false><<<grid, lbt::kThreads, 0, s>>>(init, n, n_outputs, out);
    LBT_HIP(hipGetLastError());
  }
  return LBT_OK;
}

int lbt_predict(void* stream, const void* X, int32_t x_dtype, int64_t n_rows, int32_t n_features,
                int32_t n_trees, const double* const* leaf, const int32_t* const* feature,
                const double* const* split, const int32_t* tree_nodes, int32_t n_outputs,
                double* out, void* workspace, size_t workspace_bytes)
{
  return lbt_predict_from(stream, X, x_dtype, n_rows, n_features, n_trees, leaf, feature, split, tree_nodes, n_outputs, nullptr,
                          out, workspace, workspace_bytes);
}

int lbt_pack_ensemble(void* stream, int32_t x_dtype, int32_t n_features, int32_t n_trees,
                      const double* const* leaf, const int32_t* const* feature, const double* const* split,
                      const int32_t* tree_nodes, int32_t n_outputs, void* buffer, size_t buffer_bytes,
                      lbt_packed_ensemble* ensemble)
{
  LBT_REQUIRE(ensemble != nullptr, "null ensemble descriptor");
  *ensemble = lbt_packed_ensemble{};
  LBT_REQUIRE(x_dtype == LBT_F32 || x_dtype == LBT_F64, "unsupported X dtype %d", x_dtype);
  LBT_REQUIRE(n_features >= 1 && n_outputs >= 1 && n_trees >= 1, "bad shape");
  LBT_REQUIRE(leaf && feature && split && tree_nodes, "null tree arrays");
  for (int i = 0; i < n_trees; i++)
    LBT_REQUIRE(leaf[i] && feature[i] && split[i] && tree_nodes[i] >= 1, "tree %d is incomplete", i);
  if (buffer == nullptr) {
    lbt::set_error("null buffer for the packed ensemble");
    return LBT_ERR_WORKSPACE;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (x_dtype == LBT_F32)
    LBT_TRY(lbt::pack_tiled<float>(s, n_features, n_trees, leaf, feature, split, tree_nodes, n_outputs, buffer,
                                   buffer_bytes, ensemble));
  else
    LBT_TRY(lbt::pack_tiled<double>(s, n_features, n_trees, leaf, feature, split, tree_nodes, n_outputs, buffer,
                                    buffer_bytes, ensemble));
  if (ensemble->data == nullptr) {
    lbt::set_error("ensemble does not fit the packed form (more than 16383 features, a tree of more than 65535 "
                   "nodes or too large for the LDS, or rows too wide for the LDS): use lbt_predict");
    return LBT_ERR_UNSUPPORTED;
  }
  return LBT_OK;
}

int lbt_predict_packed(void* stream, const void* X, int32_t x_dtype, int64_t n_rows, int32_t n_features,
                       const lbt_packed_ensemble* ensemble, double* out)
{
  LBT_REQUIRE(ensemble != nullptr && ensemble->data != nullptr, "ensemble was not packed");
  LBT_REQUIRE(x_dtype == ensemble->x_dtype && n_features == ensemble->n_features,
              "X (dtype %d, %d features) does not match the packed ensemble (dtype %d, %d features)", x_dtype,
              n_features, ensemble->x_dtype, ensemble->n_features);
  LBT_REQUIRE((ensemble->lanes == 4 || ensemble->lanes == 8 || ensemble->lanes == 16) && ensemble->n_trees >= 1 &&
                ensemble->n_batches >= 1 && ensemble->n_batches <= ensemble->n_trees &&
                ensemble->n_outputs >= 1 && ensemble->n_outputs <= 65535 &&
                ensemble->total_nodes >= ensemble->n_trees && ensemble->lds_bytes >= 16 &&
                static_cast<size_t>(ensemble->lds_bytes) <= lbt::kTileLds,
              "corrupt ensemble descriptor");
  LBT_REQUIRE(ensemble->bytes >= lbt_predict_workspace_bytes(ensemble->n_trees, ensemble->total_nodes,
                                                             ensemble->n_outputs, ensemble->x_dtype),
              "corrupt ensemble descriptor (buffer size)");
  if (n_rows < 1) return LBT_OK;
  LBT_REQUIRE(X && out, "null X or output");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (x_dtype == LBT_F32) return lbt::run_tiled<float>(s, static_cast<const float*>(X), n_rows, *ensemble, out);
  return lbt::run_tiled<double>(s, static_cast<const double*>(X), n_rows, *ensemble, out);
}

size_t lbt_predict_workspace_bytes(int32_t n_trees, int64_t total_nodes, int32_t n_outputs, int32_t x_dtype)
{
  if (n_trees < 0 || total_nodes < 0 || n_outputs < 1 || (x_dtype != LBT_F32 && x_dtype != LBT_F64)) return 0;
  return lbt::packed_bytes(n_trees, total_nodes, n_outputs,
                           x_dtype == LBT_F32 ? sizeof(lbt::PackedNode<float>) : sizeof(lbt::PackedNode<double>));
}

size_t lbt_predict_rows_workspace_bytes(int64_t n_rows, int32_t n_features, int32_t n_trees, const int32_t* tree_nodes,
                                        int32_t n_outputs, int32_t x_dtype)
{
  if (n_rows < 0 || n_features < 1 || n_trees < 0 || (n_trees > 0 && tree_nodes == nullptr)) return 0;
  int64_t total = 0;
  for (int i = 0; i < n_trees; i++) {
    if (tree_nodes[i] < 1) return 0;
    total += tree_nodes[i];
  }
  const size_t packed = lbt_predict_workspace_bytes(n_trees, total, n_outputs, x_dtype);
  if (packed == 0) return 0;
  const size_t ranked = lbt::ranked_workspace_bytes(n_rows, n_features, n_trees, tree_nodes, n_outputs, x_dtype);
  return ranked == 0 ? packed : ((packed + 255) & ~size_t(255)) + ranked;
}

size_t lbt_update_tree_workspace_bytes(int64_t n_rows, int32_t n_outputs, int32_t n_nodes)
{
  (void)n_rows;
  if (n_outputs < 1 || n_nodes < 1) return 0;
  return static_cast<size_t>(n_nodes) * n_outputs * 2 * sizeof(double) + 512;
}

int lbt_update_tree_rows(void* stream, const void* X, int32_t x_dtype, int64_t n_rows, int32_t n_features,
                         const double* g, const double* h, int32_t n_outputs, const int32_t* feature,
                         const double* split, int32_t n_nodes, double l1_regularization, double l2_regularization,
                         double* leaf_out, double* hessian_out, int32_t* row_leaf, void* workspace,
                         size_t workspace_bytes)
{
  LBT_REQUIRE(x_dtype == LBT_F32 || x_dtype == LBT_F64, "unsupported X dtype %d", x_dtype);
  LBT_REQUIRE(n_rows >= 0 && n_features >= 1 && n_outputs >= 1 && n_nodes >= 1, "bad shape");
  LBT_REQUIRE(feature && split && leaf_out && hessian_out, "null tree pointer");
  LBT_REQUIRE(n_rows == 0 || (X && g && h), "null input");
  if (!workspace || workspace_bytes < lbt_update_tree_workspace_bytes(n_rows, n_outputs, n_nodes)) {
    lbt::set_error("workspace missing or too small for lbt_update_tree");
    return LBT_ERR_WORKSPACE;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  uintptr_t raw = (reinterpret_cast<uintptr_t>(workspace) + 255) & ~uintptr_t(255);
  double* G     = reinterpret_cast<double*>(raw);
  lbt::UpdateArgs a;
  a.n_rows = n_rows; a.F = n_features; a.K = n_outputs; a.n_nodes = n_nodes;
  a.g = g; a.h = h; a.feature = feature; a.split = split;
  a.G = G; a.H = G + static_cast<int64_t>(n_nodes) * n_outputs; a.row_leaf = row_leaf;
  lbt::ProfScope ps(LBT_PROF_OTHER, s);
  return x_dtype == LBT_F32
           ? lbt::update_impl(s, static_cast<const float*>(X), a, l1_regularization, l2_regularization, leaf_out, hessian_out)
           : lbt::update_impl(s, static_cast<const double*>(X), a, l1_regularization, l2_regularization, leaf_out, hessian_out);
}

int lbt_update_tree(void* stream, const void* X, int32_t x_dtype, int64_t n_rows, int32_t n_features, const double* g,
                    const double* h, int32_t n_outputs, const int32_t* feature, const double* split, int32_t n_nodes,
                    double l1_regularization, double l2_regularization, double* leaf_out, double* hessian_out,
                    void* workspace, size_t workspace_bytes)
{
  return lbt_update_tree_rows(stream, X, x_dtype, n_rows, n_features, g, h, n_outputs, feature, split, n_nodes,
                              l1_regularization, l2_regularization, leaf_out, hessian_out, nullptr, workspace,
                              workspace_bytes);
}

}  // extern "C"
