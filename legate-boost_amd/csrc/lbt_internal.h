// Internal declarations shared by the translation units of liblbtree.so.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdarg>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../../include/lbtree.h"

namespace lbt {

// ---------------------------------------------------------------- errors

void set_error(const char* fmt, ...);

#define LBT_HIP(call)                                                                  \
  do {                                                                                 \
    hipError_t e__ = (call);                                                           \
    if (e__ != hipSuccess) {                                                           \
      ::lbt::set_error("%s failed: %s (%s:%d)", #call, hipGetErrorString(e__), __FILE__, \
                       __LINE__);                                                      \
      return LBT_ERR_HIP;                                                              \
    }                                                                                  \
  } while (0)

#define LBT_REQUIRE(cond, ...)          \
  do {                                  \
    if (!(cond)) {                      \
      ::lbt::set_error(__VA_ARGS__);    \
      return LBT_ERR_INVALID;           \
    }                                   \
  } while (0)

#define LBT_TRY(expr)            \
  do {                           \
    int rc__ = (expr);           \
    if (rc__ != LBT_OK) return rc__; \
  } while (0)

// ---------------------------------------------------------------- workspace

// Bump allocator over the caller's scratch buffer. In "measure" mode it only
// adds up sizes, so the same code path computes lbt_*_workspace_bytes.
struct Arena {
  char* base   = nullptr;
  size_t cap   = 0;
  size_t used  = 0;
  bool measure = false;
  bool failed  = false;

  template <typename T>
  T* take(size_t n)
  {
    size_t bytes = (n * sizeof(T) + 255) & ~size_t(255);
    size_t at    = used;
    used += bytes;
    if (measure) return nullptr;
    if (used > cap) {
      failed = true;
      return nullptr;
    }
    return reinterpret_cast<T*>(base + at);
  }
};

// ---------------------------------------------------------------- profiling

struct ProfSpan {
  int cls;
  int level;  // tree level for histogram spans, else -1
  double bytes;
  hipEvent_t start, stop;
};

// Per-level counts of one lbt_build_tree call on their way to the host: the call copies them
// into pinned memory in stream order and does not have to wait for them.
struct LevelCounts {
  long long tiles;  // tile count and padding of the device-side record
  long long instances, built_instances, built_nodes;
};
struct ProfLevels {
  LevelCounts* host;    // pinned, 64 entries
  hipEvent_t arrived;   // recorded behind the copy
  int levels;
  double bytes_per_built_row;
  double bytes_per_built_node;
  double root_extra_bytes;
};

struct Profiler {
  int mode = 0;  // 0 off, 1 every kernel class, 2 the two histogram-stage classes only
  lbt_profile acc{};
  std::vector<ProfSpan> open;  // spans not yet read back
  std::vector<hipEvent_t> pool;  // events waiting to be reused
  std::vector<ProfLevels> levels;        // level counts not yet read back
  std::vector<LevelCounts*> level_pool;  // pinned buffers waiting to be reused
  // nullptr if no pinned buffer or event can be had
  ProfLevels* begin_levels(int n_levels, double per_row, double per_node, double root_extra);
  bool wants(int cls) const
  {
    return mode == 1 || (mode == 2 && (cls == LBT_PROF_HISTOGRAM || cls == LBT_PROF_BINNING));
  }
  void begin(int cls, int level, double bytes, hipStream_t s);
  void end(hipStream_t s);
  void collect();  // waits for what the recorded events mark, then adds everything up
};
Profiler& profiler();

struct ProfScope {
  hipStream_t s;
  bool on;
  ProfScope(int cls, hipStream_t stream, double bytes = 0.0, int level = -1) : s(stream)
  {
    on = profiler().wants(cls);
    if (on) profiler().begin(cls, level, bytes, s);
  }
  ~ProfScope()
  {
    if (on) profiler().end(s);
  }
};

// ---------------------------------------------------------------- host-side state
//
// What a host thread keeps between calls, besides its error string: pinned buffers and events
// that would cost more to create per call than the calls they serve. Created on first use by
// the thread that calls lbt_build_tree, released by lbt_release_thread_resources() on that
// thread (or never: a thread that ends without calling it leaves them to the process's end).
struct ThreadResources {
  int device = 0;  // the device the handles below were created on
  // what the host reads back in the middle of a build (bin counts per feature, the quantiser's
  // overflow flag): [4 + capacity] ints, two 64-bit statistics first
  int32_t* mirror        = nullptr;
  size_t mirror_capacity = 0;
  hipEvent_t counts_here = nullptr, stats_here = nullptr;
  // staging buffer of the small tables a build sends to the device, and the event behind its copy
  char* stage           = nullptr;
  size_t stage_bytes    = 0;
  hipEvent_t stage_free = nullptr;
  // two pinned words in which kernels report to the host (see DeviceAnswer), and the last call's tag
  unsigned long long* answer = nullptr;
  uint32_t answer_tag        = 0;
};
ThreadResources& thread_resources();
// the same after making sure that what it holds belongs to the current device
int thread_resources_here(ThreadResources** out);
int release_thread_resources();

// What the builders without a wait in their middle have to learn from the device: two words of the thread's
// pinned memory that kernels early in the queue write, each (tag << 32) | value: words[0] flags (1: the
// data need the other builder, 2: a rounded value does not fit 32 bits), words[1] the number of bins.
// The host waits for them once everything is queued; the tag tells one call's answer from another's. All builds
// of a thread share the words, on whatever streams, and lbt_release_thread_resources frees them: no call
// returns while a store of its own is still to come. wait() sees both words, and a call that ends without
// it drains its stream.
struct DeviceAnswer {
  unsigned long long* words = nullptr;
  uint32_t tag              = 0;
  hipStream_t stream        = nullptr;
  bool due                  = false;  // a kernel may still store them
  int open(hipStream_t on);
  // the flags have come and say that this builder's levels are not wanted (false as long as they are out)
  bool declined() const
  {
    const unsigned long long w = *static_cast<volatile const unsigned long long*>(words);
    return (w >> 32) == tag && (w & 0xffffffffULL) != 0;
  }
  // flags: receives bit 0; bit 1 is returned as LBT_ERR_UNSUPPORTED. n_bins: null when not wanted.
  int wait(unsigned* flags, int32_t* n_bins);
  DeviceAnswer() = default;
  DeviceAnswer(const DeviceAnswer&) = delete;
  DeviceAnswer& operator=(const DeviceAnswer&) = delete;
  ~DeviceAnswer();
};

// ---------------------------------------------------------------- device math

#define LBT_M 2147483647u
#define LBT_A 48271u

// Reduction modulo the Mersenne prime m = 2^31 - 1 of a value below 2^62:
// 2^31 == 1 (mod m), so the high part can be folded onto the low part.
__host__ __device__ inline uint32_t mod_m(uint64_t p)
{
  p = (p & LBT_M) + (p >> 31);
  p = (p & LBT_M) + (p >> 31);
  return static_cast<uint32_t>(p >= LBT_M ? p - LBT_M : p);
}
// thrust::minstd_rand seeding: s mod m, 1 if that is 0.
__host__ __device__ inline uint32_t minstd_seed(uint32_t s)
{
  uint32_t x = mod_m(s);
  return x == 0 ? 1u : x;
}
__host__ __device__ inline uint32_t minstd_next(uint32_t x)
{
  return mod_m(static_cast<uint64_t>(x) * LBT_A);
}
__host__ __device__ inline uint32_t minstd_discard(uint32_t x, uint64_t z)
{
  uint64_t mult = LBT_A, acc = 1;
  while (z > 0) {
    if (z & 1) acc = mod_m(acc * mult);
    mult = mod_m(mult * mult);
    z >>= 1;
  }
  return mod_m(static_cast<uint64_t>(x) * acc);
}
// n / d from an approximate reciprocal r of d (a relative error of 2^-23 is enough): two steps of Newton's iteration, then the remainder's
// correction. The bits of the division where no intermediate value leaves the normal range (tests/test_quotients.py).
__host__ __device__ inline double quotient_from(double n, double d, double r)
{
  r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
  r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
  const double q = n * r;
  return __builtin_fma(__builtin_fma(-d, q, n), r, q);
}

// thrust::uniform_real_distribution<double>(0,1) on one raw draw.
__host__ __device__ inline double uniform01(uint32_t draw)
{
  // the quotient by 2147483646, correctly rounded for every draw (tests/test_quotients.py): the product with its reciprocal and the
  // remainder's correction, eight instructions less than a division
  constexpr double d = 2147483646.0, r = 1.0 / d;
  const double n = static_cast<double>(draw - 1u), q = n * r;
  return __builtin_fma(__builtin_fma(-d, q, n), r, q);
}

// fmix64 on a signed 64-bit value: arithmetic right shifts, wrapping multiplies
// (reference: build_tree.cu:143-154).
__host__ __device__ inline int64_t hash64(int64_t k)
{
  k ^= k >> 33;
  k = static_cast<int64_t>(static_cast<uint64_t>(k) * 0xff51afd7ed558ccdULL);
  k ^= k >> 33;
  k = static_cast<int64_t>(static_cast<uint64_t>(k) * 0xc4ceb9fe1a85ec53ULL);
  k ^= k >> 33;
  return k;
}
__host__ __device__ inline int64_t hash_combine1(int64_t seed, int64_t v)
{
  uint64_t sum = static_cast<uint64_t>(hash64(v)) + 0x9e3779b9ULL +
                 (static_cast<uint64_t>(seed) << 6) + static_cast<uint64_t>(seed >> 2);
  return seed ^ static_cast<int64_t>(sum);
}
// seed of the stochastic rounding of (row, output): build_tree.cu:190, :353
__host__ __device__ inline int64_t gpair_seed(int64_t seed, int64_t row, int64_t output)
{
  return hash_combine1(hash_combine1(seed, row), output);
}

// build_tree.h:106-121
__host__ __device__ inline double leaf_gain(double grad, double hess, double l1, double reg)
{
  double z = 0.0;
  if (grad > l1) {
    z = grad - l1;
  } else if (grad < -l1) {
    z = grad + l1;
  }
  return (z * z) / (hess + reg);
}
// build_tree.h:123-137
__host__ __device__ inline double calculate_gain(double gl, double hl, double gr, double hr,
                                                 double gp, double hp, double l1, double reg,
                                                 double min_split_gain)
{
  return (0.5 * (leaf_gain(gl, hl, l1, reg) + leaf_gain(gr, hr, l1, reg) -
                 leaf_gain(gp, hp, l1, reg))) -
         min_split_gain;
}
// build_tree.h:139-152
__host__ __device__ inline double calculate_leaf_value(double G, double H, double l1, double l2)
{
  double z = 0.0;
  if (G > l1) {
    z = G - l1;
  } else if (G < -l1) {
    z = G + l1;
  }
  return -z / (H + l2);
}

// legateboost.py:209-211: weight, learning rate, least hessian
constexpr double kMinHessian = 1e-8;
__device__ inline void weigh(double g0, double h0, double w, double lr, double* g, double* h)
{
  *g = (g0 * w) * lr;
  *h = fmax(h0 * w, kMinHessian);
}

// build_tree.h:64-74
__host__ __device__ inline int parent_of(int i) { return (i - 1) / 2; }
__host__ __device__ inline int left_child(int i) { return 2 * i + 1; }
__host__ __device__ inline int right_child(int i) { return 2 * i + 2; }
__host__ __device__ inline int sibling_of(int i) { return (i % 2 == 0) ? i - 1 : i + 1; }
inline int64_t level_begin(int l) { return (int64_t(1) << l) - 1; }
inline int64_t level_end(int l) { return (int64_t(1) << (l + 1)) - 1; }

struct I64Pair {
  int64_t grad;
  int64_t hess;
};

// build_tree.h:76-104; node_sums is [max_nodes][K] pairs, output 0 decides.
__device__ inline bool compute_histogram_bin(int node, const I64Pair* node_sums, int K,
                                             bool parent_histogram_exists)
{
  if (node == 0) return true;
  if (node < 0) return false;
  if (!parent_histogram_exists) return true;
  int parent = parent_of(node);
  int l = left_child(parent), r = right_child(parent);
  int64_t hl = node_sums[static_cast<int64_t>(l) * K].hess;
  int64_t hr = node_sums[static_cast<int64_t>(r) * K].hess;
  int histogram_node = (hl < hr) ? l : r;
  return histogram_node == node;
}

// Lets `kernel` use up to `bytes` of dynamic LDS. The attribute belongs to the device the
// function is loaded on, so it is set once per device; `done` is the caller's per-kernel record
// (one flag per device ordinal). Setting it twice from two threads is harmless.
constexpr int kMaxDevices = 64;
template <typename KernelT>
int allow_dynamic_lds(KernelT kernel, size_t bytes, std::atomic<bool> (&done)[kMaxDevices])
{
  int device = 0;
  LBT_HIP(hipGetDevice(&device));
  if (device >= 0 && device < kMaxDevices && done[device].load(std::memory_order_acquire)) return LBT_OK;
  LBT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(bytes)));
  if (device >= 0 && device < kMaxDevices) done[device].store(true, std::memory_order_release);
  return LBT_OK;
}

inline int ceil_div(int64_t a, int64_t b) { return static_cast<int>((a + b - 1) / b); }

__device__ inline void atomic_add_i64(int64_t* p, int64_t v)
{
  atomicAdd(reinterpret_cast<unsigned long long*>(p), static_cast<unsigned long long>(v));
}

// The histogram buffer: [node - node_begin][K][B] pairs (build_tree.h:231-306).
struct HistView {
  I64Pair* data;
  int node_begin;
  int node_end;
  int K;
  int B;
  // One byte per node, where the level's histograms are what the rows add up to, whatever the reference leaves
  // unscanned above it (see build_tree_impl); else null. Set: the node's own histogram is not.
  const uint8_t* tainted;
  __device__ bool contains(int node) const { return node >= node_begin && node < node_end; }
  __device__ I64Pair* at(int node, int k, int bin) const
  {
    return data + ((static_cast<int64_t>(node - node_begin) * K + k) * B + bin);
  }
  // Whether rows are added to the node's histogram (else it is its parent's without its sibling's)
  __device__ bool builds(int node, const I64Pair* node_sums) const
  {
    const int parent = parent_of(node);
    if (tainted != nullptr && node > 0 && contains(parent) && tainted[parent] != 0) return true;
    return compute_histogram_bin(node, node_sums, K, contains(parent));
  }
};

// ---------------------------------------------------------------- histogram stage

// Written by the tile planner for one batch of nodes.
struct LevelMeta {
  int32_t n_tiles;
  int32_t pad;
  long long instances;        // rows held by the nodes of the batch
  long long built_instances;  // rows whose node's histogram is built
  long long built_nodes;
};


// Where the records of one histogram feature group live in the bin cache. A record is what
// one row contributes to the group: the feature-relative bins of the group's features, zero
// bytes up to zero_end, and (single-output trees) the row's packed (grad, hess) pair at q_off.
struct RecInfo {
  int64_t base;      // byte offset of row 0's record
  int32_t in_row;    // of them, from the first byte of row 0 of its plane (see hist_prepare)
  int32_t stride;    // bytes between the records of consecutive rows (multiple of 32)
  int32_t size;      // bytes of one record (multiple of 32)
  int32_t q_off;     // byte offset of the int2 (grad, hess) inside a record, or -1
  int32_t zero_end;  // bytes [bins_end, zero_end) of a record are zero
  int32_t bins_end;  // bytes of bins in a record
};

// Per-tree state of the histogram stage (see lbt_histogram.hip).
struct HistSetup {
  int n_features     = 0;
  int n_groups       = 0;   // histogram feature groups (LDS holds a group's packed sub-histogram)
  int n_sgroups      = 0;   // search feature groups (LDS holds proposals and lookup tables)
  int vec            = 1;   // features per lane of the search (1, 2 or 4)
  int cells          = 0;   // table entries per feature (power of two)
  int search_steps   = 0;   // ceil(log2(max bins of a feature + 1))
  size_t lds_bytes   = 0;   // LDS of the search / binning kernel
  bool is_f64        = false;
  // device buffers (carved from the caller's workspace)
  int32_t* groups    = nullptr;  // [n_groups + 1]
  int32_t* sgroups   = nullptr;  // [n_sgroups + 1]; the same array as groups when the cache is off
  // lookup tables and cell functions of the search (see build_cells_kernel)
  uint2* tables      = nullptr;  // [2][n_features][cells / 32]: one entry per 32 cells
  void* map_x        = nullptr;  // X dtype [2][n_features][2]
  float* map_t       = nullptr;  // [n_features][2]
  int32_t* straight  = nullptr;  // [n_features]
  int32_t* tile_start = nullptr;
  int4* tiles         = nullptr;  // one descriptor per tile of the batch in flight
  LevelMeta* meta    = nullptr;
  int32_t* pair_sync = nullptr;  // kPairSyncSlots arrival counters of the root launch's row ranges
  // sub-histograms parked for the reduction pass: slot s holds partial_stride packed bins
  unsigned long long* partials = nullptr;
  // the slots of list t = (node of the batch) * groups * outputs + group * outputs + output:
  // partial_lists[t * kPartialListCap ..], partial_list_count[t] of them
  int32_t* partial_lists = nullptr;
  int32_t* partial_list_count = nullptr;  // [kPartialMaxLists]
  int32_t* partial_count = nullptr;  // slots handed out by the running launch
  int partial_slots = 0;
  int partial_stride = 0;
  // bin cache: written by the root binning pass and read by the histogram kernel of every
  // level instead of X; a row's records lie side by side, [row][histogram group][record], in a plane per search group of the
  // pass where its groups are whole histogram groups (RecInfo)
  void* binned         = nullptr;  // null: cache off
  size_t binned_capacity = 0;      // bytes available at `binned`
  int bin_bytes        = 0;        // 1 or 2
  bool ragged          = false;    // binning pass: rows are no whole number of lane vectors (or start unaligned)
  int bvec             = 1;        // cached bins a lane of the histogram kernel loads at once
  bool embed           = false;    // records carry the row's (grad, hess)
  size_t blds_bytes    = 0;        // LDS of the histogram kernel (packed sub-histogram only)
  int stripe_log       = -1;       // log2 of the striped layout's row width in features; negative: [feature][bin]
  int stripe_bins      = 0;        // bins of the widest feature (rows of the striped array)
  int even_lanes       = 0;        // lanes per row shared by all groups of a histogram launch; 0: per group
  int spread           = 0;        // bins a lane takes of a row where four lanes share them evenly (Stripes::per); 0: they do not
  RecInfo* rec         = nullptr;  // [n_groups]
  int64_t max_rec_stride = 0;      // widest row of a plane, bytes
  int64_t row_bytes      = 0;      // bytes of a row in all planes
  int pieces           = 0;        // 16-byte pieces of bins of a row's records
  int max_bins         = 0;        // bins of the widest feature
  int share            = 0;        // lanes that share a record in the binning pass, 0: each has words of its own (share_of_record)
  int2* bin_lanes      = nullptr;  // [bin_lanes_max] lanes of a row in the binning pass (see bin_lanes)
  // feature-major copy of the bins, [feature][row], written by the root histogram launch for the
  // position updates (null: not wanted)
  void* bins_t           = nullptr;
  int64_t bins_t_stride  = 0;      // elements between consecutive features (multiple of 128)
  // the part of the workspace that holds groups, sgroups, bin_lanes and rec
  // (and nothing else): hist_prepare fills it with one copy
  void* upload_block   = nullptr;
  size_t upload_bytes  = 0;
  int rpp              = 0;        // rows per workgroup pass, search / binning kernel
  int brpp             = 0;        // rows per workgroup pass, histogram kernel on cached bins
};

constexpr int kMaxCells = 16384;  // table cells per feature at most (one entry of 8 bytes per 32 cells)
constexpr int kPairSyncSlots = 4096;
// bins of the widest feature group that fits the LDS beside the lanes' spare slots
constexpr int kPartialStrideMax = (160 * 1024 - 512 - 4096 - 8 * 1024) / 8;
constexpr int kPartialSlots = 1024;      // sub-histograms one launch can park
constexpr int kPartialListCap = 320;      // slots one list can index (a node's row ranges plus overflow merges)
constexpr int kPartialMaxLists = 4096;   // (node, group, output) triples the reduction pass is launched for
constexpr int kHistThreads       = 1024;
// LDS a histogram-stage workgroup may fill; 4 KB of the 160 KB stay free for the tile window
constexpr size_t kLdsBudget = 160 * 1024 - 512 - 4096;

// Upper bound on the cache bytes one row can take for n_features features with at most
// split_samples bins each: the bins plus, per histogram group, the embedded gradient pair,
// alignment and padding to the 32-byte record pitch. The group count is bounded through the
// fewest features a group can hold.
inline int64_t bin_row_bytes_max(int n_features, int split_samples)
{
  const int bin_bytes = split_samples <= 256 ? 1 : 2;
  int64_t cap = static_cast<int64_t>((kLdsBudget - 8 * kHistThreads) / (8 * static_cast<size_t>(split_samples)));
  if (cap >= 4) cap = cap / 4 * 4;
  if (cap < 1) cap = 1;
  // one more for the uneven widths of a balanced split, two more that may be taken to fill idle CUs
  const int64_t groups_max = (n_features + cap - 1) / cap + 3;
  return static_cast<int64_t>(n_features) * bin_bytes + groups_max * 48;
}

// ... and the cache as a whole: at most a plane per feature, each starting on a multiple of kPlaneAlign bytes
constexpr int kPlaneAlign = 128;
// entries of HistSetup::bin_lanes: a lane per four features, up to 13 and two for each group, which has four features or more (up to
// three features: a lane each)
inline size_t bin_lanes_max(int n_features) { return 4 * static_cast<size_t>(n_features) + 16; }
inline size_t bin_cache_bytes(int64_t n_rows, int n_features, int split_samples)
{
  return static_cast<size_t>(n_rows * bin_row_bytes_max(n_features, split_samples)) + static_cast<size_t>(kPlaneAlign) * n_features;
}

struct HistBatch {
  const void* X;
  int F;
  const int2* qgh;
  int K;
  const int32_t* rows;  // row numbers in node order (the level's segments index into it)
  const int32_t* seg;
  int j0;
  int n_nodes;
  int level_first;
  const void* proposals;
  const int32_t* row_pointers;
  const int32_t* bin_feature;  // [bins] feature of every proposal
  HistView hist;
  const unsigned long long* qstats;
  const I64Pair* node_sums;
  LevelMeta* level_total;
  int64_t n_rows;
  bool fill_cache;  // run the binning pass first (the bin cache does not hold this X and these proposals yet)
  bool identity;    // rows[i] == i for every i (the root of a tree that starts from the original order)
  bool planned = false;  // the tiles have been planned (hist_plan)
};

// Which nodes of a batch are built, and their tiles (plan_tiles_block)
struct PlanArgs {
  int j0, j1, level_first;
  const int32_t* seg;
  const I64Pair* node_sums;
  HistView hist;
  int tile_rows;
  int4* tiles;
  LevelMeta* meta;
  LevelMeta* level_total;
  int32_t* pair_sync;
  int32_t* partial_count;
  int32_t* partial_list_count;
  int blocks;  // workgroups of kPlanThreads
};
constexpr int kPlanThreads = 256;
// What plans a batch below the root in a launch of the caller's; blocks: 0 where hist_launch has to do it.
int hist_plan(const HistSetup& hs, const HistBatch& b, PlanArgs* plan);

// What else begins with the tables: the root's outputs (build_tree.cu:1175-1185), the quantiser's two words for the host, and
// histograms to clear.
struct RootArgs {
  double* leaf;
  const I64Pair* node_sums;
  int K;
  const double* scales;
  double l1, l2;
  const unsigned long long* qstats;
  unsigned long long* host_stats;
  uint4* clear;
  int64_t n16;
};
// Chooses groups / table size from the host copy of the row pointers and builds
// the tables on the device. root: optional
int hist_prepare(hipStream_t stream, HistSetup& hs, bool is_f64, int F, int K, int64_t n_rows,
                 const std::vector<int32_t>& rp, const void* proposals, const int32_t* row_pointers,
                 const void* X, const RootArgs* root = nullptr);
// Plans tiles for the batch and launches the histogram kernel.
int hist_launch(hipStream_t stream, const HistSetup& hs, const HistBatch& b, int depth);

// A level whose histograms stay in the LDS (see lbt_direct_level.hip).
struct Cand;
constexpr int kDirectMaxBins = 512;  // of a feature: 32 KB of LDS per workgroup
struct DirectLevel {
  int level_first, n_nodes, n_features, n_groups;
  int64_t n_rows;
  const void* binned;
  const RecInfo* rec;
  const int32_t* groups;
  const int32_t* rows;
  const int32_t* seg;
  const int32_t* block_seg;  // node that holds position b * slab (-1: a row that has stopped)
  int slab;
  int range;                  // positions that a workgroup takes of a large node (direct_range)
  unsigned long long* large;  // histograms of large nodes, direct_large_bytes, all zero between nodes and levels
  int32_t* arrivals;          // ... of which counters (set by direct_level_launch)
  const int32_t* row_pointers;
  const uint8_t* feature_set;
  const double* scales;
  double l1, l2, min_split_gain;
  const double* proposals;
  I64Pair* node_sums;
  Cand* partial;   // [n_nodes][n_features] best split of a feature
  I64Pair* left;   // and its left sums
  double* leaf;
  int32_t* feature;
  double* split;
  double* gain;
  int32_t* split_bin;
};
int direct_range(const HistSetup& hs, int64_t n_rows, size_t room);  // 0: the large nodes' histograms have no room
size_t direct_large_bytes(const HistSetup& hs, int64_t n_rows, int range);  // multiple of 16
int direct_level_launch(hipStream_t stream, DirectLevel a, const HistSetup& hs);

// ---------------------------------------------------------------- builder for few rows
// (lbt_small_tree.hip)

constexpr int kSmallMaxRows    = 8192;
constexpr int kSmallMaxOutputs = 16;
constexpr int kSmallMaxDepth   = 13;

struct SmallCand {
  double gain;
  uint32_t key;  // order among equal gains, larger wins; 0: no candidate
  int32_t rel;   // bin of the feature (the builder for medium sizes keeps a flag with it)
};

// Device buffers of a build, carved from the caller's workspace.
constexpr int kSmallDecideFeatures = 64;  // a lane each of the wave that decides a node

struct SmallTreeState {
  int64_t pitch;          // elements between the rows of a feature and those of the next (multiple of 8)
  uint32_t* order[2];     // [F][pitch] row | bin << 16 by (node, bin); the order of level d is order[d & 1]
  uint16_t* bins;         // [F][pitch] bin of every row
  double* proposals;      // [F][S]
  int32_t* counts;        // [F] proposals
  int32_t* rp;            // [F] first bin of the feature among all bins
  uint16_t* node_of_pos[2];  // [pitch] node of the level that holds a place of the order, 0xffff: a leaf's; the root's in the first one
  uint8_t* code;          // [N] side a row of a split node takes: 1 left, 2 right
  int2* seg;              // [max_nodes] places of a node's rows: the first one, and how many
  int32_t* live;          // [max_depth + 1] the level has nodes
  I64Pair* base;          // [max_nodes][K] sums of the rows in front of the node's places
  I64Pair* node_sums;     // [max_nodes][K]
  int2* qgh;              // [N][K]
  double* scales;         // [4]
  SmallCand* cand[2];     // [nodes of a level][F]
  I64Pair* left[2];       // the same: what lies left of a candidate; null where no scan decides the level above it
  // all levels in one launch (else null): see small_levels_kernel
  uint32_t* sync;             // [kSmallDecideFeatures]
  unsigned long long* found;  // [inner nodes][3][F]
};
bool small_tree_levels_fit(int64_t N, int F, int K, int max_depth);
bool small_tree_fits(int64_t N, int F, int K, int max_depth, int S);
// n_bins: receives the number of bins of all features (null: not wanted). level_totals: [max_depth], added
// to (null: not wanted).
// *taken: the tree has been queued; false (with LBT_OK): the data need the other builder, which has to
// write every output again.
template <typename T>
int small_tree_build(hipStream_t stream, const SmallTreeState& st, const T* X, int64_t row_offset, int64_t N, int F,
                     int K, const double* g, const double* h, const uint8_t* feature_set, const lbt_build_params& prm,
                     double* leaf, int32_t* feature, double* split, double* gain, double* hessian, int32_t* row_leaf,
                     int32_t* n_bins, LevelMeta* level_totals, bool* taken);

// ---------------------------------------------------------------- builder for medium sizes
// (lbt_mid_tree.hip)

constexpr int kMidMaxDepth      = 10;
constexpr int kMidMaxLevelNodes = 1 << (kMidMaxDepth - 1);
constexpr int kMidMaxOutputs    = 16;
constexpr int64_t kMidMaxValues = int64_t(200) * 1000 * 1000;

struct MidTreeState {
  int64_t pitch;          // elements between features, outputs (multiple of 256, at least the rows)
  int bin_bytes;          // 1 or 2
  void* bins;             // [F][pitch]
  void* props;            // X dtype [F][S]
  double* proposals;      // [F][S] the same
  int cells;              // cell functions and tables of the bin search, [F] each (see build_cells_kernel)
  uint2* tables;          // [F][cells / 32]
  void* map_x;            // X dtype [F][2]
  float* map_t;           // [F][2]
  int32_t* counts;        // [F]
  int32_t* rp;            // [F + 1]
  double* chunk_sums;     // [2][chunks of 4096 entries]
  int2* q;                // [K][pitch]
  uint16_t* row_node[2];  // [pitch] node of the level, 0xffff: none; of the root in the first one
  unsigned long long* q_stats;  // [4] sum of the positive rounded grads, of the negative ones, flags
  unsigned long long* images;   // packed histograms of the row ranges
  uint2* hist[2];         // scanned histograms, lower halves of grad and hess, [node][K][F][S]; level d in hist[d & 1]
  uint2* left;            // [nodes of the last level][F] the same of what lies left of a feature's best split (one output)
  I64Pair* node_sums;     // [max_nodes][K]
  double* scales;         // [4]
  SmallCand* cand;        // [nodes of a level][F]
  int2* splits;           // [nodes of a level]
  int32_t* live;          // [max_depth + 1]
};
bool mid_tree_fits(int64_t N, int F, int K, int max_depth, int S);
bool mid_beats_small(int64_t N, int F, int K, int max_depth, int S);
// Bytes from hist[0] on: hist[0], hist[1] and images, one behind the other.
size_t mid_hist_bytes(int64_t N, int F, int K, int max_depth, int S);
// As small_tree_build.
template <typename T>
int mid_tree_build(hipStream_t stream, const MidTreeState& st, const T* X, int64_t row_offset, int64_t N, int F, int K,
                   const double* g, const double* h, const uint8_t* feature_set, const lbt_build_params& prm,
                   double* leaf, int32_t* feature, double* split, double* gain, double* hessian, int32_t* row_leaf,
                   int32_t* n_bins, LevelMeta* level_totals, bool* taken);

}  // namespace lbt
