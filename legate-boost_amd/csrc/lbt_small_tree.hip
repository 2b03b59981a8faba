// BuildTreeTask for inputs of few rows: 2 launches, or 1 + 2 * max_depth, instead of about ten per level.
//
// The builder of lbt_build_tree.hip is made for rows by the million. With a few thousand of them its
// launches do almost nothing (5 us each, about 90 for a tree of depth 8) and its histograms are
// mostly empty: 128 nodes x 500 features x 256 bins for 5,000 rows. Here no histogram exists. Every
// feature keeps the rows sorted by (node, bin of that feature); the running sums along that order
// are the scanned histogram at its occupied bins (build_tree.cu:597-668), and a bin without rows
// has the sums, and with them the gain, of the last occupied bin before it.
//
//   small_prologue_kernel   one workgroup per feature: split proposals (build_tree.cu:867-964), the bin of
//                           every row, the rows sorted by bin; one workgroup: quantiser and root
//                           (build_tree.cu:51-204, 1154-1187); the rest clear the outputs
//   small_scan_kernel       one workgroup per feature and level: carries its order over to the level
//                           (a stable partition inside every node), running sums, gains, and the best
//                           split of the feature per node (build_tree.cu:682-740)
//   small_levels_kernel     one output, up to 64 features and 4096 rows, trees that are not too deep: all scans and decisions in one launch,
//                           one workgroup per feature
//   small_apply_kernel      one workgroup per node and level: best feature, the node's outputs and its
//                           children (build_tree.cu:740-782), the side of each of its rows. Where a level has few
//                           candidates every scan workgroup of the next one does that for itself (a launch less)
//
// The sums are integers, so they do not depend on the order of rows; gains and leaf values are formed
// by the same functions from the same sums as in the other builder: the trees are identical. One rule of
// the reference needs the histogram itself: a running sum that is positive in neither half leaves the bin
// unscanned (build_tree.cu:645). That matters only if some row has a non-positive rounded hessian and a
// pair other than (0, 0); the prologue reports such rows, the levels behind it then do nothing, and the caller
// takes the other builder.
#include <algorithm>
#include <limits>
#include <type_traits>

#include "lbt_device.h"
#include "lbt_internal.h"

namespace lbt {
namespace {

constexpr int kPrologueThreads = 1024;
constexpr int kNone            = 0xffff;  // node_of_pos of a row whose node did not split
constexpr int kQuantChunks     = 8;       // chunks of 4096 entries the quantiser's workgroup takes
constexpr unsigned long long kNotFound = ~0ull;  // neither bits of a gain, nor a key and a bin, nor sums of hessians (see small_levels_kernel)

struct PrologueArgs {
  int64_t row_offset;
  int N, F, K, S;
  int32_t seed;
  int64_t dataset_rows;
  const double* g;
  const double* h;
  const double* first_level;  // the quantiser's chunk sums if the caller has them, else null
  double l1, l2;
  int64_t max_nodes;
  int max_depth;
  double* leaf;
  int32_t* feature;
  double* split;
  double* gain;
  double* hessian;
  unsigned long long* answer;  // pinned host memory (see DeviceAnswer)
  uint32_t tag;
};

// Quantiser, root sums and root outputs: the arithmetic and the order of sums of sum_chunk,
// find_scales and quantise_kernel (lbt_build_tree.hip), for at most kQuantChunks chunks.
__device__ inline void small_quantise(const PrologueArgs& a, const SmallTreeState& st, unsigned char* smem)
{
  double* s_a = reinterpret_cast<double*>(smem);           // [4][256]
  double* s_b = s_a + 1024;                                 // [4][256]
  double* s_chunk_a = s_b + 1024;                           // [kQuantChunks]
  double* s_chunk_b = s_chunk_a + kQuantChunks;
  double* s_scale   = s_chunk_b + kQuantChunks;             // [4]
  unsigned long long* s_sum = reinterpret_cast<unsigned long long*>(s_scale + 4);  // [2 * K]
  __shared__ unsigned s_flags;
  const int n = a.N * a.K;
  const int m = (n + 4095) / 4096;
  const int quarter = threadIdx.x >> 8, t = threadIdx.x & 255;
  if (threadIdx.x == 0) s_flags = 0;
  for (int i = threadIdx.x; i < 2 * a.K; i += kPrologueThreads) s_sum[i] = 0;
  if (threadIdx.x < kQuantChunks) s_chunk_a[threadIdx.x] = s_chunk_b[threadIdx.x] = 0.0;
  __syncthreads();
  if (a.first_level != nullptr) {
    if (static_cast<int>(threadIdx.x) < m) {
      s_chunk_a[threadIdx.x] = a.first_level[threadIdx.x];
      s_chunk_b[threadIdx.x] = a.first_level[m + threadIdx.x];
    }
    __syncthreads();
  } else {
    // four chunks at a time, 256 threads each
    for (int c0 = 0; c0 < m; c0 += 4) {
      const int c = c0 + quarter;
      double xa = 0.0, xb = 0.0;
      // four at a time without a branch around the loads: behind one, each is waited for before the next is asked for
      for (int j0 = 0; j0 < 16 && c * 4096 + 256 * j0 < n; j0 += 4) {
        double ga[4], ha[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int e = min(c * 4096 + t + 256 * (j0 + j), n - 1);
          ga[j] = a.g[e];
          ha[j] = a.h[e];
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const bool in = c * 4096 + t + 256 * (j0 + j) < n;
          xa += in ? fabs(ga[j]) : 0.0;
          xb += in ? fabs(ha[j]) : 0.0;
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
      if (t == 0 && c < m) {
        s_chunk_a[c] = s_a[quarter * 256];
        s_chunk_b[c] = s_b[quarter * 256];
      }
      __syncthreads();
    }
  }
  if (threadIdx.x == 0) {
    // the second level's tree over at most kQuantChunks sums; the lanes past them add zeros
    for (int stride = kQuantChunks / 2; stride >= 1 && m > 1; stride >>= 1)
      for (int i = 0; i < stride; i++) {
        s_chunk_a[i] += s_chunk_a[i + stride];
        s_chunk_b[i] += s_chunk_b[i + stride];
      }
    const double max_int = 2147483647.0;
    const double sg = s_chunk_a[0] == 0 ? 1 : max_int / s_chunk_a[0];
    const double sh = s_chunk_b[0] == 0 ? 1 : max_int / s_chunk_b[0];
    s_scale[0] = sg;
    s_scale[1] = sh;
    s_scale[2] = 1.0 / sg;
    s_scale[3] = 1.0 / sh;
  }
  __syncthreads();
  const double sg = s_scale[0], sh = s_scale[1];
  int64_t sum_g = 0, sum_h = 0;  // single output
  unsigned flags = 0;
  for (int e = threadIdx.x; e < n; e += kPrologueThreads) {
    const int row = a.K == 1 ? e : e / a.K, k = a.K == 1 ? 0 : e - row * a.K;
    const double grad = a.g[e], hess = a.h[e];
    int64_t qg, qh;
    quantise_pair(grad, hess, sg, sh, static_cast<int64_t>(a.seed), row + a.row_offset, k, &qg, &qh);
    if (qg > 2147483647LL || qg < -2147483647LL || qh > 2147483647LL || qh < -2147483647LL) flags |= 2u;
    if (qh <= 0 && (qg != 0 || qh != 0)) flags |= 1u;
    st.qgh[e] = make_int2(static_cast<int>(qg), static_cast<int>(qh));
    if (a.K == 1) {
      sum_g += qg;
      sum_h += qh;
    } else {
      atomicAdd(&s_sum[k], static_cast<unsigned long long>(qg));
      atomicAdd(&s_sum[a.K + k], static_cast<unsigned long long>(qh));
    }
  }
  if (a.K == 1) {
    sum_g = wave_inclusive_sum(sum_g);
    sum_h = wave_inclusive_sum(sum_h);
    if ((threadIdx.x & 63) == 63) {
      atomicAdd(&s_sum[0], static_cast<unsigned long long>(sum_g));
      atomicAdd(&s_sum[1], static_cast<unsigned long long>(sum_h));
    }
  }
  if (flags != 0) atomicOr(&s_flags, flags);
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(a.answer, (static_cast<unsigned long long>(a.tag) << 32) | s_flags, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  if (threadIdx.x < 4) st.scales[threadIdx.x] = s_scale[threadIdx.x];
  for (int k = threadIdx.x; k < a.K; k += kPrologueThreads) {
    const I64Pair ns{static_cast<int64_t>(s_sum[k]), static_cast<int64_t>(s_sum[a.K + k])};
    st.node_sums[k] = ns;
    st.base[k]      = I64Pair{0, 0};
    a.leaf[k]       = calculate_leaf_value(static_cast<double>(ns.grad) * s_scale[2],
                                           static_cast<double>(ns.hess) * s_scale[3], a.l1, a.l2);
    a.hessian[k]    = static_cast<double>(ns.hess) * s_scale[3];
  }
  if (threadIdx.x == 0) {
    a.feature[0]    = -1;
    a.split[0]      = 0.0;
    a.gain[0]       = 0.0;
    st.seg[0]       = make_int2(0, a.N);
    st.live[0]      = s_flags == 0 ? 1 : 0;  // data for the other builder: the levels that are queued have nothing to do
  }
}

// Proposals, bins and the order of one feature.
template <typename T>
__device__ inline void small_feature(const T* __restrict__ X, const PrologueArgs& a, const SmallTreeState& st, int f,
                                     unsigned char* smem)
{
  int P = 1;
  while (P < a.S) P <<= 1;
  // the proposals' scratch, then counts (places) of the bins and the rows in order
  int* s_count      = reinterpret_cast<int*>(smem + static_cast<size_t>(P) * kProposalScratch<T>);  // [P + 1]
  uint32_t* s_order = reinterpret_cast<uint32_t*>(s_count + P + 4);                                  // [N]
  __shared__ int s_wave[kPrologueThreads / 64];
  const int tid = threadIdx.x;
  for (int i = tid; i <= P; i += kPrologueThreads) s_count[i] = 0;
  // the feature's values, asked for before the samples they are searched among (past the last row: its value again)
  T x[kSmallMaxRows / kPrologueThreads];
#pragma unroll
  for (int u = 0; u < kSmallMaxRows / kPrologueThreads; u++)
    x[u] = X[static_cast<int64_t>(min(tid + u * kPrologueThreads, a.N - 1)) * a.F + f];
  const SampleSpec sp{a.S, a.seed, a.dataset_rows, a.row_offset, a.N, a.F};
  const T* s_prop = nullptr;
  const int n     = feature_proposals<T, kPrologueThreads>(X, sp, f, P, smem, s_wave, &s_prop);
  for (int i = tid; i < n; i += kPrologueThreads)
    st.proposals[static_cast<int64_t>(f) * a.S + i] =
      i == n - 1 ? std::numeric_limits<double>::infinity() : static_cast<double>(s_prop[i]);
  if (tid == 0) st.counts[f] = n;
  // bins: the number of proposals below the value, the last one never being below
  uint16_t* bins = st.bins + static_cast<int64_t>(f) * st.pitch;
  int my_bin[kSmallMaxRows / kPrologueThreads];
#pragma unroll
  for (int u = 0; u < kSmallMaxRows / kPrologueThreads; u++) {
    const int r = tid + u * kPrologueThreads;
    my_bin[u]   = -1;
    if (r < a.N) {
      int lo = 0, len = n - 1;
      while (len > 0) {
        const int half = len >> 1;
        const bool go  = s_prop[lo + half] < x[u];
        lo             = go ? lo + half + 1 : lo;
        len            = go ? len - half - 1 : half;
      }
      my_bin[u] = lo;
      bins[r]   = static_cast<uint16_t>(lo);
      atomicAdd(&s_count[lo], 1);
    }
  }
  __syncthreads();
  // counting sort of the rows by bin (an entry of the order is row | bin << 16); which of a bin's rows comes first does not matter
  const int c0 = 2 * tid < n ? s_count[2 * tid] : 0, c1 = 2 * tid + 1 < n ? s_count[2 * tid + 1] : 0;
  const int place = block_exclusive_sum32<kPrologueThreads>(c0 + c1, s_wave);
  if (2 * tid < n) s_count[2 * tid] = place;
  if (2 * tid + 1 < n) s_count[2 * tid + 1] = place + c0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kSmallMaxRows / kPrologueThreads; u++)
    if (my_bin[u] >= 0)
      s_order[atomicAdd(&s_count[my_bin[u]], 1)] = static_cast<uint32_t>(tid + u * kPrologueThreads) |
                                                   (static_cast<uint32_t>(my_bin[u]) << 16);
  __syncthreads();
  uint32_t* order = st.order[0] + static_cast<int64_t>(f) * st.pitch;
  for (int i = tid; i < a.N; i += kPrologueThreads) order[i] = s_order[i];
}

// The i-th of F features by XCD: workgroups 8 apart run on one XCD and take features side by side, so that a row's cache lines are
// read by one L2 (an eighth of 5000 x 500 doubles fits it) and not by all eight.
__device__ __forceinline__ int feature_by_xcd(int i, int F)
{
  const int x = i & 7;
  return x * (F >> 3) + min(x, F & 7) + (i >> 3);
}

// Bound by the latency of a feature's column (a line per value) and of the searches behind it. 5000 x 500 doubles: 46.7 us with features
// dealt to the XCDs in turn, 74 registers (one workgroup to a CU) and a wait for every 1024 rows; 31.4 with features by XCD,
// two workgroups to a CU (eight waves a SIMD) and all rows asked for at the start. 1000 x 10: 11.9 and 11.6.
template <typename T>
__global__ void __launch_bounds__(kPrologueThreads, 8)
  small_prologue_kernel(const T* __restrict__ X, PrologueArgs a, SmallTreeState st)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int block = blockIdx.x;
  if (block == 0) {
    small_quantise(a, st, smem_raw);
    return;
  }
  if (block <= a.F) {
    small_feature<T>(X, a, st, feature_by_xcd(block - 1, a.F), smem_raw);
    return;
  }
  // the outputs of every node but the root, and what the levels count on being zero
  const int64_t stride = static_cast<int64_t>(gridDim.x - 1 - a.F) * kPrologueThreads;
  const int64_t first  = static_cast<int64_t>(block - 1 - a.F) * kPrologueThreads + threadIdx.x;
  for (int64_t i = first; i < a.max_nodes * a.K; i += stride)
    if (i >= a.K) {
      a.leaf[i]    = 0.0;
      a.hessian[i] = 0.0;
    }
  for (int64_t i = first; i < a.max_nodes; i += stride)
    if (i >= 1) {
      a.feature[i]    = -1;
      a.split[i]      = 0.0;
      a.gain[i]       = 0.0;
      st.seg[i] = make_int2(0, 0);
    }
  for (int64_t i = first; i < a.N; i += stride) st.node_of_pos[0][i] = 0;
  if (first >= 1 && first <= a.max_depth) st.live[first] = 0;
  if (st.sync != nullptr) {
    if (first < kSmallDecideFeatures) st.sync[first] = 0;
    const int64_t words = 3 * ((int64_t(1) << a.max_depth) - 1) * a.F;
    for (int64_t i = first; i < words; i += stride) st.found[i] = kNotFound;
  }
}

struct LevelArgs {
  int N, F, K, S;
  int depth;
  int level_first;  // first node of the level; its node j is level_first + j
  int n_nodes;
  bool last;        // no further level follows
  const uint16_t* node_in;  // [pitch] node of this level (scan that decides: of the level above) that holds a place
  uint16_t* node_out;       // scan that decides: of this level
  const SmallCand* cand_above;   // scan that decides: what the level above found, [node][F]
  const I64Pair* left_above;     // and what lies left of it
  SmallCand* cand;          // what this level finds
  I64Pair* left;            // null: small_apply_kernel follows
  int lanes_log;            // scan that decides: lanes per node of the level above, log2
  bool all_bins;            // scan that decides: the bins of all features lie in the LDS
  double* leaf;
  int32_t* feature;
  double* split;
  double* gain;
  double* hessian;
  int32_t* row_leaf;
  unsigned long long* n_bins;  // pinned host memory: the number of all bins (see DeviceAnswer)
  uint32_t tag;
  const uint8_t* feature_set;
  double l1, l2, min_split_gain;
};

// Consecutive values of one thread, kE of them from an address aligned to 16 bytes (16-bit values: to
// their size).
template <int kE>
__device__ __forceinline__ void load_u16(const uint16_t* p, int (&out)[kE])
{
  static_assert(kE == 2 || kE == 4 || kE == 8, "4, 8 or 16 bytes per thread");
  uint32_t w[kE / 2];
  if constexpr (kE == 2) {
    w[0] = *reinterpret_cast<const uint32_t*>(p);
  } else if constexpr (kE == 4) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    w[0] = v.x, w[1] = v.y;
  } else {
    const uint4 v = *reinterpret_cast<const uint4*>(p);
    w[0] = v.x, w[1] = v.y, w[2] = v.z, w[3] = v.w;
  }
#pragma unroll
  for (int i = 0; i < kE / 2; i++) {
    out[2 * i]     = w[i] & 0xffff;
    out[2 * i + 1] = w[i] >> 16;
  }
}
template <int kE>
__device__ __forceinline__ void load_u32(const uint32_t* p, uint32_t (&out)[kE])
{
  if constexpr (kE == 2) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    out[0] = v.x, out[1] = v.y;
  }
#pragma unroll
  for (int i = 0; i < kE / 4; i++) {
    const uint4 v = reinterpret_cast<const uint4*>(p)[i];
    out[4 * i] = v.x, out[4 * i + 1] = v.y, out[4 * i + 2] = v.z, out[4 * i + 3] = v.w;
  }
}

template <int kE>
__device__ __forceinline__ void store_u32(uint32_t* p, const uint32_t (&v)[kE])
{
  if constexpr (kE == 2) *reinterpret_cast<uint2*>(p) = make_uint2(v[0], v[1]);
#pragma unroll
  for (int i = 0; i < kE / 4; i++) reinterpret_cast<uint4*>(p)[i] = make_uint4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
}

// Where a split falls among equal gains of a node (cand_better): the largest bin mod 512, counted over all
// bins, then the smallest bin. Bins [bin, next) of the feature, of which only the first has rows, share a
// gain; one of them is 511 mod 512, or their residues ascend. Larger keys win, none is 0.
__device__ __forceinline__ unsigned tie_key(int rp, int bin, int next)
{
  const int pick = min((rp + bin) | 511, rp + next - 1);
  return (static_cast<unsigned>(pick & 511) << 11 | static_cast<unsigned>(2047 - (pick - rp))) + 1u;
}

// Places of the order a scan workgroup holds, by rows, and the LDS it then asks for at a level of n_nodes nodes
// (see small_scan_kernel). 156 KB of the 160 leave room for its static arrays (0.6 KB).
constexpr size_t kScanLds = 156 * 1024;
__host__ __device__ constexpr int small_scan_places(int64_t N) { return N <= 1024 ? 1024 : N <= 2048 ? 2048 : N <= 4096 ? 4096 : kSmallMaxRows; }
__host__ __device__ constexpr size_t small_scan_lds(int64_t N, int64_t n_nodes)
{
  return static_cast<size_t>((N + 1) / 2 * 2 * 8 + (small_scan_places(N) + 4) * 4 + n_nodes * 12 + (n_nodes / 2 + 1) * 4 +
                             (N + 3) / 4 * 4 + 16);
}

// The LDS a launch asks for: the order takes the rows and what 16-byte accesses may touch behind them.
__host__ __device__ constexpr int64_t small_scan_order(int64_t N) { return (N + 15) / 8 * 8; }
__host__ __device__ constexpr size_t small_scan_use(int64_t N, int64_t n_nodes)
{
  return static_cast<size_t>((N + 1) / 2 * 2 * 8 + small_scan_order(N) * 4 + n_nodes * 12 + (n_nodes / 2 + 1) * 4 + (N + 3) / 4 * 4 + 31) / 16 * 16;
}

// What a scan that decides needs beside that, of the level above.
constexpr int kDecidePasses = 2;   // candidates a thread looks at
constexpr int decide_loads(int threads) { return threads == 1024 ? 4 : 8; }   // 16-byte pieces of all features' bins it stages
constexpr int kDecideRows  = 4096;  // rows up to which a scan decides: with eight places a thread it gained nothing
constexpr int kDecideLanes = 4;  // log2 of the fewest lanes a node takes

// The largest value of an aligned group of 16, 32 or 64 lanes, in all of them
__device__ __forceinline__ unsigned group_max_u32(unsigned v, int lanes_log)
{
  auto take = [&](auto ctrl) {
    const unsigned o = static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), decltype(ctrl)::value, 0xf, 0xf, true));
    v = o > v ? o : v;
  };
  take(std::integral_constant<int, 0x128>{});  // the lanes of a row of 16, turned by 8, 4, 2 and 1
  take(std::integral_constant<int, 0x124>{});
  take(std::integral_constant<int, 0x122>{});
  take(std::integral_constant<int, 0x121>{});
  if (lanes_log > 4) v = max(v, static_cast<unsigned>(__shfl_xor(static_cast<int>(v), 16, 64)));
  if (lanes_log > 5) v = max(v, static_cast<unsigned>(__shfl_xor(static_cast<int>(v), 32, 64)));
  return v;
}
__host__ __device__ constexpr size_t small_decide_use(int64_t n_nodes) { return static_cast<size_t>((n_nodes / 2 + 2) / 2 * 2 * (16 + 8 + 8 + 8 + 4) + 16 + 16); }

// kT threads take kE consecutive places of the order each (kT * kE >= N). What a place needs of its row
// (its pair of the first output, its side) is staged in the LDS in row order: gathered from the L2 these
// are three scattered accesses per place, and a workgroup's 8192 places then take a level 90 us
// (5,000 rows x 500 features). Everything that does not depend on another load is asked for first: the
// levels of a small tree are a chain of memory latencies. So the nodes' sums, the parents' terms of the gain and the
// segments are staged too where the LDS has the room (kStaged): looked up in memory whenever a thread's places
// pass on to another node, they are a latency per node (1000 x 10, depth 8: 9.2 us a launch, with that and the
// gains below 7.8).
// kG: places of a thread whose gains are formed side by side (one output). A place's two quotients are a chain of 400
// cycles or more, and one place after the other was half of the launch on 1000 x 10. With more features than CUs it is
// the other way round: 64 registers let two workgroups of 1024 threads share a CU, and one place at a time is enough
// (5000 x 500: 32 us a launch, now 25; with 66 registers it was one workgroup).
// kDecides: the level above has been scanned, not decided. Every workgroup finds all its splits (a candidate per lane), sums
// of its children and sides of its rows for itself, feature 0's writes them down. A launch of small_apply_kernel was a third of
// a level (1000 x 10, depth 8: 4.5 of 12.4 us and the gap in front of it). Fits with such launches and without, us: 1000 x 10 f64,
// depth 8, 12 rounds 1580 and 1290; 2000 x 16, depth 8, 5 rounds 815 and 720; 4000 x 8, depth 6 860 and 740; 1000 x 40, depth 8 740
// and 665; 3000 x 60, depth 7 900 and 850. From 4096 rows on (8000 x 30, 7000 x 12, 5000 x 64) it gained nothing.
// kLeft: the next scan may decide, so what lies left of a node's best split goes with it (the scans that decide always have
// it). 2500 x 150, whose scans never decide: 12.0 us a launch with it, 11.2 without.
template <int kT, int kE, bool kSingle, int kG, bool kStaged, bool kDecides, bool kLeft = kDecides>
__global__ void __launch_bounds__(kT, kT == 1024 && kG == 1 && kSingle ? 8 : 1)
  small_scan_kernel(SmallTreeState st, LevelArgs a)
{
  static_assert(!(kDecides || kLeft) || (kSingle && kStaged && kG > 1), "one output, nodes in the LDS");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  int2* s_q                  = reinterpret_cast<int2*>(smem_raw);               // [N]
  uint32_t* s_order          = reinterpret_cast<uint32_t*>(s_q + (a.N + 1) / 2 * 2);  // [small_scan_order(N)]
  unsigned long long* s_gain = reinterpret_cast<unsigned long long*>(s_order + small_scan_order(a.N));  // [n_nodes] bits of the best gain
  unsigned* s_key            = reinterpret_cast<unsigned*>(s_gain + a.n_nodes);  // [n_nodes] its place in the order of ties
  int* s_left_before         = reinterpret_cast<int*>(s_key + a.n_nodes);        // [n_nodes / 2 + 1]
  uint8_t* s_code            = reinterpret_cast<uint8_t*>(s_left_before + a.n_nodes / 2 + 1);  // [N]
  I64Pair* s_ns              = reinterpret_cast<I64Pair*>(smem_raw + small_scan_use(a.N, a.n_nodes));  // kStaged: [n_nodes]
  I64Pair* s_base            = s_ns + a.n_nodes;
  double* s_parent           = reinterpret_cast<double*>(s_base + a.n_nodes);
  int2* s_seg                = reinterpret_cast<int2*>(s_parent + a.n_nodes);
  const int n_pad            = (a.n_nodes / 2 + 2) / 2 * 2;
  I64Pair* s_left_above      = reinterpret_cast<I64Pair*>(s_seg + a.n_nodes);    // kDecides, of the level above: [n_pad]
  int2* s_split              = reinterpret_cast<int2*>(s_left_above + n_pad);
  int2* s_seg_above          = s_split + n_pad;
  double* s_gain_above       = reinterpret_cast<double*>(s_seg_above + n_pad);
  int* s_left_behind         = reinterpret_cast<int*>(s_gain_above + n_pad);
  uint16_t* s_bins           = reinterpret_cast<uint16_t*>(s_left_behind + (n_pad + 3) / 4 * 4);  // all_bins: [F][pitch]
  __shared__ I64Pair s_pair[2][kT / 64];
  __shared__ int s_wave[kT / 64];
  __shared__ int s_rp;
  const int f = blockIdx.x, tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int i0   = tid * kE;
  const bool usable = a.feature_set == nullptr || a.feature_set[f] != 0;
  SmallCand* const out = a.cand + f;  // node j: out[j * F]
  const uint32_t* order_in = st.order[a.depth == 0 ? 0 : (a.depth - 1) & 1] + static_cast<int64_t>(f) * st.pitch;
  // Places, rows and nodes past the last one are asked for as the last one: hipcc keeps a load that only some lanes ask for
  // behind a branch, and waits for its answer before the next branch (1000 x 10, scans that decide: 23,000 cycles each, 17,000
  // without such waits). With eight places a thread many threads have none, and what they ask for costs more.
  constexpr bool kClamped = kE <= 4;
  uint32_t entry[kE];
  int node[kE], node_next = kNone;
  if constexpr (kClamped) {
    const int i_in = min(i0, static_cast<int>(st.pitch) - kE);
    load_u32<kE>(order_in + i_in, entry);
    load_u16<kE>(a.node_in + i_in, node);
    node_next = a.node_in[min(i0 + kE, a.N - 1)];
  } else {
#pragma unroll
    for (int e = 0; e < kE; e++) {
      entry[e] = 0;
      node[e]  = kNone;
    }
    if (i0 < a.N) {
      load_u32<kE>(order_in + i0, entry);
      load_u16<kE>(a.node_in + i0, node);
      if (i0 + kE < a.N) node_next = a.node_in[i0 + kE];
    }
  }
  const int live = st.live[kDecides ? a.depth - 1 : a.depth];
  int rp         = a.depth == 0 ? 0 : st.rp[f];  // first bin of the feature among all bins
  const double inv_g = st.scales[2], inv_h = st.scales[3];
  const double reg   = 1e-5 > a.l2 ? 1e-5 : a.l2;
  // kDecides: what the level above has left, a candidate per lane and pass, a node per thread. (All that a workgroup
  // reads is asked for before the first answer is waited for: what another XCD wrote takes 3000 cycles to arrive.)
  constexpr int kPasses = kDecides ? kDecidePasses : 1, kLoads = kDecides ? decide_loads(kT) : 1;
  const int above_first = (a.level_first - 1) / 2, n_above = a.n_nodes / 2, sub = tid & ((1 << a.lanes_log) - 1);
  SmallCand cand_of[kPasses];
  // (Members of their own: hipcc keeps an array of pairs in scratch memory, and what goes there is waited for at once. These
  // launches took 9.0 us on 1000 x 10 that way, now 8.5; 14.5 and 13.8 on 4000 x 8.)
  int64_t left_grad[kPasses], left_hess[kPasses];
  I64Pair ns_above{0, 0}, base_above{0, 0};
  int2 seg_of{0, 0};
  uint4 bins_of[kLoads];
  const int n16 = a.all_bins ? a.F * static_cast<int>(st.pitch / 8) : 1;
  if constexpr (kDecides) {
#pragma unroll
    for (int p = 0; p < kPasses; p++) {
      const int j  = min((p * kT + tid) >> a.lanes_log, n_above - 1), at = j * a.F + min(sub, a.F - 1);
      cand_of[p]   = a.cand_above[at];
      const I64Pair left_of = a.left_above[at];
      left_grad[p] = left_of.grad;
      left_hess[p] = left_of.hess;
    }
    const int above = above_first + min(tid, n_above - 1);
    ns_above        = st.node_sums[above];
    base_above      = st.base[above];
    seg_of          = st.seg[above];
#pragma unroll
    for (int u = 0; u < kLoads; u++) bins_of[u] = reinterpret_cast<const uint4*>(st.bins)[min(tid + u * kT, n16 - 1)];
  }
  // all loads are under way before the first is stored: a loop that loads and stores waits once per turn
  int2 pair[kSingle && kG > 1 ? kE : 1];
  if constexpr (kSingle && kG > 1) {
#pragma unroll
    for (int u = 0; u < kE; u++)
      if (kClamped || tid + u * kT < a.N) pair[u] = st.qgh[min(tid + u * kT, a.N - 1)];
  } else if (kSingle && usable) {
    for (int i = tid; i < a.N; i += kT) s_q[i] = st.qgh[i];
  }
  static_assert(kE >= 4 || kDecides, "sides of four rows at a time");
  uint32_t code[(kE + 3) / 4];
  if (!kDecides && kClamped && a.depth > 0) {
#pragma unroll
    for (int u = 0; u < kE / 4; u++) code[u] = *reinterpret_cast<const uint32_t*>(st.code + min(4 * (tid + u * kT), static_cast<int>(st.pitch) - 4));
  }
  if (!kClamped) {
#pragma unroll
    for (int u = 0; u < kE / 4; u++)
      if (a.depth > 0 && 4 * (tid + u * kT) < a.N) code[u] = *reinterpret_cast<const uint32_t*>(st.code + 4 * (tid + u * kT));
  }
  if (kStaged && kSingle && !kDecides && usable)
    for (int j = tid; j < a.n_nodes; j += kT) {
      const I64Pair ns = st.node_sums[a.level_first + j];
      s_base[j]        = st.base[a.level_first + j];
      s_seg[j]         = st.seg[a.level_first + j];
      s_ns[j]          = ns;
      s_parent[j]      = leaf_gain(static_cast<double>(ns.grad) * inv_g, static_cast<double>(ns.hess) * inv_h, a.l1, reg);
    }
  if constexpr (kSingle && kG > 1) {
#pragma unroll
    for (int u = 0; u < (kClamped ? kE : 0); u++) arrived(pair[u]);
#pragma unroll
    for (int u = 0; u < kE; u++)
      if (tid + u * kT < a.N) s_q[tid + u * kT] = pair[u];
  }
#pragma unroll
  for (int u = 0; u < kE / 4; u++)
    if (!kDecides && a.depth > 0 && 4 * (tid + u * kT) < a.N) *reinterpret_cast<uint32_t*>(s_code + 4 * (tid + u * kT)) = code[u];
  if (live == 0 && a.depth > 0) return;
  // (kDecides, feature 0's workgroup) what follows from the splits of the level above, when there is nothing else to do
  double split_value = 0.0;  // thread j: of node j
  auto write_outputs = [&]() {
    const int j = tid;
    if (f != 0 || j >= a.n_nodes / 2 || s_split[j].x < 0) return;
    a.feature[above_first + j] = s_split[j].x;
    a.split[above_first + j]   = split_value;
    a.gain[above_first + j]    = s_gain_above[j];
    for (int side = 0; side < 2; side++) {
      const double g = static_cast<double>(s_ns[2 * j + side].grad) * inv_g, h = static_cast<double>(s_ns[2 * j + side].hess) * inv_h;
      a.leaf[a.level_first + 2 * j + side]    = calculate_leaf_value(g, h, a.l1, a.l2);
      a.hessian[a.level_first + 2 * j + side] = h;
    }
  };
  if constexpr (kDecides) {
#pragma unroll
    for (int u = 0; u < kLoads; u++) arrived(bins_of[u]);
    arrived(seg_of);
    if (tid < n_above) s_seg_above[tid] = seg_of;
#pragma unroll
    for (int u = 0; u < kLoads; u++)
      if (tid + u * kT < n16) reinterpret_cast<uint4*>(s_bins)[tid + u * kT] = bins_of[u];
#pragma unroll
    for (int p = 0; p < kPasses; p++) {
      if ((p * kT) >> a.lanes_log < n_above) {
        // gains are not negative: their bits compare as whole numbers, upper halves first
        const int j        = (p * kT + tid) >> a.lanes_log;
        const uint64_t own = static_cast<uint64_t>(__double_as_longlong(cand_of[p].gain));
        const unsigned own_hi = static_cast<unsigned>(own >> 32), own_lo = static_cast<unsigned>(own);
        const unsigned own_key = sub < a.F ? cand_of[p].key : 0u;  // (a copy of the last feature's is none)
        const unsigned hi  = group_max_u32(own_hi, a.lanes_log);
        const unsigned lo  = group_max_u32(own_hi == hi ? own_lo : 0u, a.lanes_log);
        const unsigned key = group_max_u32(own_hi == hi && own_lo == lo ? own_key : 0u, a.lanes_log);
        const double best  = __longlong_as_double(static_cast<int64_t>(static_cast<uint64_t>(hi) << 32 | lo));
        const bool splits  = key != 0 && best > 1e-5;
        if (j < n_above) {
          if (!splits && sub == 0) s_split[j] = make_int2(-1, 0);
          if (splits && sub < a.F && own_hi == hi && own_lo == lo && own_key == key) {  // (keys of different candidates differ: one lane)
            s_split[j]      = make_int2(sub, cand_of[p].rel);
            s_gain_above[j] = best;
            s_left_above[j].grad = left_grad[p];
            s_left_above[j].hess = left_hess[p];
          }
        }
      }
    }
    __syncthreads();
    const bool keeps = usable || f == 0;  // this feature's order
    if (f == 0 && tid < n_above && s_split[tid].x >= 0)
      split_value = st.proposals[static_cast<int64_t>(s_split[tid].x) * a.S + s_split[tid].y];
    unsigned left = 0, goes_on = 0;
    int2 sp[kE];
    int b[kE];
#pragma unroll
    for (int e = 0; e < kE; e++) {
      sp[e] = i0 + e < a.N && node[e] != kNone ? s_split[node[e]] : make_int2(-1, 0);
      b[e]  = 0;
    }
    auto bin_at = [&](int e) { return sp[e].x * static_cast<int>(st.pitch) + static_cast<int>(entry[e] & 0xffff); };
    if (a.all_bins) {
#pragma unroll
      for (int e = 0; e < kE; e++)
        if (sp[e].x >= 0) b[e] = s_bins[bin_at(e)];
    } else if (keeps) {
#pragma unroll
      for (int e = 0; e < kE; e++)
        if (sp[e].x >= 0) b[e] = st.bins[bin_at(e)];
    }
    if (f == 0 && a.row_leaf != nullptr) {
#pragma unroll
      for (int e = 0; e < kE; e++)
        if (i0 + e < a.N && node[e] != kNone && sp[e].x < 0) a.row_leaf[entry[e] & 0xffff] = above_first + node[e];
    }
    if (tid < n_above) {
      // (thread j: children of node j; without a split they have no rows and nobody asks for them)
      const bool splits       = s_split[tid].x >= 0;
      const I64Pair left_sums = splits ? s_left_above[tid] : I64Pair{0, 0};
      const I64Pair right{ns_above.grad - left_sums.grad, ns_above.hess - left_sums.hess};
      const I64Pair base_right{base_above.grad + left_sums.grad, base_above.hess + left_sums.hess};
      s_ns[2 * tid]        = splits ? left_sums : I64Pair{0, 0};
      s_ns[2 * tid + 1]    = splits ? right : I64Pair{0, 0};
      s_base[2 * tid]      = base_above;
      s_base[2 * tid + 1]  = base_right;
      s_parent[2 * tid]    = leaf_gain(static_cast<double>(left_sums.grad) * inv_g, static_cast<double>(left_sums.hess) * inv_h, a.l1, reg);
      s_parent[2 * tid + 1] = leaf_gain(static_cast<double>(right.grad) * inv_g, static_cast<double>(right.hess) * inv_h, a.l1, reg);
    }
    if (!usable)
      for (int j = tid; j < a.n_nodes; j += kT) out[static_cast<int64_t>(j) * a.F] = SmallCand{0.0, 0u, 0};
    if (!keeps) return;
    for (int j = tid; j < a.n_nodes; j += kT) {
      s_gain[j] = 0;
      s_key[j]  = 0;
    }
#pragma unroll
    for (int e = 0; e < kE; e++) {
      goes_on |= sp[e].x >= 0 ? 1u << e : 0u;
      left |= sp[e].x >= 0 && b[e] <= sp[e].y ? 1u << e : 0u;
    }
    const int before = block_exclusive_sum32<kT>(__popc(left), s_wave);
#pragma unroll
    for (int e = 0; e < kE; e++)
      if ((goes_on >> e) & 1u) {
        const int2 at = s_seg_above[node[e]];
        if (at.x == i0 + e) s_left_before[node[e]] = before + __popc(left & ((1u << e) - 1u));
        if (at.x + at.y - 1 == i0 + e) s_left_behind[node[e]] = before + __popc(left & ((2u << e) - 1u));
      }
    const bool next_goes_on = i0 + kE < a.N && node_next != kNone && s_split[node_next].x >= 0;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kE; e++) {
      const int i = i0 + e;
      if (i < a.N) {
        int to = i, child = kNone;
        if ((goes_on >> e) & 1u) {
          const int first = s_left_before[node[e]], lefts = s_left_behind[node[e]] - first, x0 = s_seg_above[node[e]].x;
          const int l     = before + __popc(left & ((1u << e) - 1u)) - first;
          to    = (left >> e) & 1u ? x0 + l : i + lefts - l;
          child = 2 * node[e] + (i - x0 < lefts ? 0 : 1);
        }
        s_order[to] = entry[e];
        node[e]     = child;
      } else {
        node[e] = kNone;
      }
    }
    if (next_goes_on) {
      const int lefts = s_left_behind[node_next] - s_left_before[node_next];
      node_next       = 2 * node_next + (i0 + kE - s_seg_above[node_next].x < lefts ? 0 : 1);
    } else {
      node_next = kNone;
    }
    if (f == 0) {
      if (tid < n_above && s_split[tid].x >= 0) {
        const int lefts = s_left_behind[tid] - s_left_before[tid], child = a.level_first + 2 * tid;
        st.seg[child]           = make_int2(seg_of.x, lefts);
        st.seg[child + 1]       = make_int2(seg_of.x + lefts, seg_of.y - lefts);
        st.node_sums[child]     = s_ns[2 * tid];
        st.node_sums[child + 1] = s_ns[2 * tid + 1];
        st.base[child]          = s_base[2 * tid];
        st.base[child + 1]      = s_base[2 * tid + 1];
        st.live[a.depth]        = 1;
      }
#pragma unroll
      for (int e = 0; e < kE; e++)
        if (i0 + e < a.N) a.node_out[i0 + e] = static_cast<uint16_t>(node[e]);
    }
    __syncthreads();
    uint32_t* order_out = st.order[a.depth & 1] + static_cast<int64_t>(f) * st.pitch;
    if (i0 < a.N) {
      load_u32<kE>(s_order + i0, entry);
      store_u32<kE>(order_out + i0, entry);  // (entries past N are never looked at)
    }
    if (!usable) {
      write_outputs();
      return;
    }
  } else {
  if (a.depth == 0) {
    int mine = 0;
    for (int i = tid; i < f; i += kT) mine += st.counts[i];
    const int excl = block_exclusive_sum32<kT>(mine, s_wave);
    if (tid == kT - 1) {
      s_rp = st.rp[f] = excl + mine;
      if (f == a.F - 1)
        __hip_atomic_store(a.n_bins, (static_cast<unsigned long long>(a.tag) << 32) | static_cast<unsigned>(s_rp + st.counts[f]),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __syncthreads();
    if (live == 0) return;  // (the number of bins is reported all the same)
    rp = s_rp;
  }
  if (!usable) {
    for (int j = tid; j < a.n_nodes; j += kT) out[static_cast<int64_t>(j) * a.F] = SmallCand{0.0, 0u, 0};
    if (f != 0) return;  // small_apply_kernel walks the rows in feature 0's order
  }
  for (int j = tid; j < a.n_nodes; j += kT) {
    s_gain[j] = 0;
    s_key[j]  = 0;
  }
#pragma unroll
  for (int e = 0; e < kE; e++)
    if (i0 + e >= a.N) node[e] = kNone;
  if (kClamped && i0 + kE >= a.N) node_next = kNone;
  if (a.depth > 0) {
    // node[] already is the node of this level at the place: both children of a parent lie where the
    // parent's rows lay, the left one first
    int2 seg[kE];  // the left child's
    const bool from_lds = kStaged && kSingle && usable;
    if (!from_lds) {
#pragma unroll
      for (int e = 0; e < kE; e++) seg[e] = node[e] != kNone ? st.seg[a.level_first + (node[e] & ~1)] : make_int2(-1, 0);
    }
    __syncthreads();
    if (from_lds) {
#pragma unroll
      for (int e = 0; e < kE; e++) seg[e] = node[e] != kNone ? s_seg[node[e] & ~1] : make_int2(-1, 0);
    }
    unsigned left = 0;
#pragma unroll
    for (int e = 0; e < kE; e++)
      if (node[e] != kNone) left |= s_code[entry[e] & 0xffff] == 1 ? 1u << e : 0u;
    const int before = block_exclusive_sum32<kT>(__popc(left), s_wave);
#pragma unroll
    for (int e = 0; e < kE; e++)
      if (seg[e].x == i0 + e) s_left_before[node[e] >> 1] = before + __popc(left & ((1u << e) - 1u));
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kE; e++) {
      const int i = i0 + e;
      if (i < a.N) {
        int to = i;
        if (node[e] != kNone) {
          const int l = before + __popc(left & ((1u << e) - 1u)) - s_left_before[node[e] >> 1];
          to = (left >> e) & 1u ? seg[e].x + l : i + seg[e].y - l;
        }
        s_order[to] = entry[e];
      }
    }
    __syncthreads();
    uint32_t* order_out = st.order[a.depth & 1] + static_cast<int64_t>(f) * st.pitch;
    if (i0 < a.N) {
      load_u32<kE>(s_order + i0, entry);
      store_u32<kE>(order_out + i0, entry);  // (entries past N are never looked at)
    }
  } else {
    // the neighbour's first bin is looked up below
    if (i0 < a.N) s_order[i0] = entry[0];
    __syncthreads();
  }
  if (!usable) return;
  }

  // occupied bins: the places that are the last of their (node, bin); the last rows of a node leave
  // nothing on the right: never a split
  int bin[kE + 1];
#pragma unroll
  for (int e = 0; e < kE; e++) bin[e] = static_cast<int>(entry[e] >> 16);
  bin[kE] = i0 + kE < a.N ? static_cast<int>(s_order[i0 + kE] >> 16) : 0;
  unsigned ends = 0;
#pragma unroll
  for (int e = 0; e < kE; e++) {
    const int nn = e + 1 < kE ? node[e + 1] : node_next;
    if (node[e] != kNone && nn == node[e] && bin[e + 1] != bin[e]) ends |= 1u << e;
  }
  if constexpr (kSingle) {
    // A thread's places are consecutive, so its nodes come one after the other: the best split of a node
    // that begins and ends inside the thread is final, those of its first and last node meet the
    // other threads' in the LDS. Sums, parent's term and best split of the node at hand stay in registers.
    int2 q[kG > 1 ? kE : 1];
    auto pair_at = [&](int e) { return i0 + e < a.N ? s_q[entry[e] & 0xffff] : make_int2(0, 0); };
    // Sums are formed in their lower 32 bits. Absolute grads (hessians) sum up to less than 2^31 + N + 1024; with the root's sum G of them, sums
    // over any rows lie between -down and up, down = (2^31 + N + 1024 - G) / 2 + 1, up with + G, less than 2^32 apart: the lower half of
    // a sum + down is the sum + down. As doubles such whole numbers are exact.
    const I64Pair all    = st.node_sums[0];
    const int64_t most   = (int64_t(1) << 31) + a.N + 1024;
    const uint32_t down_g = static_cast<uint32_t>((most - all.grad) / 2 + 1), down_h = static_cast<uint32_t>((most - all.hess) / 2 + 1);
    const double from_g = static_cast<double>(down_g), from_h = static_cast<double>(down_h);
    uint2* const s_sums = reinterpret_cast<uint2*>(s_pair[0]);
    uint2 sum           = make_uint2(0, 0);
#pragma unroll
    for (int e = 0; e < kE; e++) {
      const int2 v = pair_at(e);
      if constexpr (kG > 1) q[e] = v;
      sum.x += static_cast<uint32_t>(v.x);
      sum.y += static_cast<uint32_t>(v.y);
    }
    const uint32_t ig = wave_inclusive_sum32(sum.x);
    const uint32_t ih = wave_inclusive_sum32(sum.y);
    if (lane == 63) s_sums[wave] = make_uint2(ig, ih);
    __syncthreads();
    uint2 run = make_uint2(ig - sum.x, ih - sum.y);
#pragma unroll 4  // (not all in registers at once)
    for (int w = 0; w < kT / 64; w++) {
      run.x += w < wave ? s_sums[w].x : 0;
      run.y += w < wave ? s_sums[w].y : 0;
    }
    int first_node = kNone, cur = kNone;
    double first_gain = 0.0, cur_gain = 0.0;
    unsigned first_key = 0, cur_key = 0;
    uint2 first_left = make_uint2(0, 0), cur_left = make_uint2(0, 0);  // with `down` added
    auto put_left = [&](int j, const uint2& left) {
      if (kLeft && a.left != nullptr)
        a.left[static_cast<int64_t>(j) * a.F + f] =
          I64Pair{static_cast<int64_t>(left.x) - static_cast<int64_t>(down_g), static_cast<int64_t>(left.y) - static_cast<int64_t>(down_h)};
    };
    // what a running sum is added to (taken from) for the sum left (right) of it in node j, with `down` added
    auto node_at = [&](int j, uint2& to_left, uint2& to_right, double& parent) {
      I64Pair ns, base;
      if constexpr (kStaged) {
        ns     = s_ns[j];
        base   = s_base[j];
        parent = s_parent[j];
      } else {
        ns     = st.node_sums[a.level_first + j];
        base   = st.base[a.level_first + j];
        parent = leaf_gain(static_cast<double>(ns.grad) * inv_g, static_cast<double>(ns.hess) * inv_h, a.l1, reg);
      }
      to_left  = make_uint2(down_g - static_cast<uint32_t>(base.grad), down_h - static_cast<uint32_t>(base.hess));
      to_right = make_uint2(down_g + static_cast<uint32_t>(base.grad) + static_cast<uint32_t>(ns.grad),
                            down_h + static_cast<uint32_t>(base.hess) + static_cast<uint32_t>(ns.hess));
    };
    auto grads  = [&](uint32_t v) { return static_cast<double>(v) - from_g; };
    auto hesses = [&](uint32_t v) { return static_cast<double>(v) - from_h; };
    // calculate_gain with the parent's term formed once per node
    const bool plain = plain_quotients(a.l1, inv_g, inv_h, reg);
    auto gain_of = [&](double lg, double lh, double rg, double rh, double parent) {
      lg *= inv_g, rg *= inv_g, lh *= inv_h, rh *= inv_h;
      if (plain) return 0.0 + ((0.5 * (quotient_plain(lg * lg, lh + reg) + quotient_plain(rg * rg, rh + reg) - parent)) - a.min_split_gain);
      return 0.0 + ((0.5 * (leaf_gain(lg, lh, a.l1, reg) + leaf_gain(rg, rh, a.l1, reg) - parent)) - a.min_split_gain);
    };
    auto next_node = [&](int j) {
      if (first_node == kNone) {
        first_node = cur;  // (kNone again while there was none before)
        first_gain = cur_gain;
        first_key  = cur_key;
        first_left = cur_left;
      } else if (cur_key != 0) {
        s_gain[cur] = static_cast<unsigned long long>(__double_as_longlong(cur_gain));
        s_key[cur]  = cur_key;
        put_left(cur, cur_left);
      }
      cur      = j;
      cur_gain = 0.0;
      cur_key  = 0;
    };
    auto offer = [&](double gain, int e, const uint2& left) {
      if (gain >= cur_gain) {
        const unsigned key = tie_key(rp, bin[e], bin[e + 1]);
        if constexpr (kLeft) {
          const bool better = gain > cur_gain || key > cur_key;
          cur_left.x        = better ? left.x : cur_left.x;
          cur_left.y        = better ? left.y : cur_left.y;
        }
        cur_key  = gain > cur_gain ? key : max(cur_key, key);
        cur_gain = gain;
      }
    };
    if constexpr (kG == 1) {
      uint2 to_left = make_uint2(0, 0), to_right = make_uint2(0, 0);
      double parent = 0.0;
#pragma unroll
      for (int e = 0; e < kE; e++) {
        const int2 v = pair_at(e);
        run.x += static_cast<uint32_t>(v.x);
        run.y += static_cast<uint32_t>(v.y);
        if ((ends >> e) & 1u) {
          if (node[e] != cur) {
            next_node(node[e]);
            node_at(cur, to_left, to_right, parent);
          }
          const uint2 ls  = make_uint2(run.x + to_left.x, run.y + to_left.y);
          const double lh = hesses(ls.y), rh = hesses(to_right.y - run.y);
          if (lh > 0 && rh > 0) {
            const double gain = gain_of(grads(ls.x), lh, grads(to_right.x - run.x), rh, parent);
            if (gain > 0) offer(gain, e, ls);
          }
        }
      }
    } else {
#pragma unroll
      for (int e0 = 0; e0 < kE; e0 += kG) {
        double gain[kG];
        bool wanted[kG];
        uint2 left_of[kG];
#pragma unroll
        for (int u = 0; u < kG; u++) {
          const int e = e0 + u;
          run.x += static_cast<uint32_t>(q[e].x);
          run.y += static_cast<uint32_t>(q[e].y);
          uint2 to_left, to_right;
          double parent;
          node_at(node[e] != kNone ? node[e] : 0, to_left, to_right, parent);
          const uint2 ls  = make_uint2(run.x + to_left.x, run.y + to_left.y);
          const double lh = hesses(ls.y), rh = hesses(to_right.y - run.y);
          wanted[u]  = ((ends >> e) & 1u) != 0 && lh > 0 && rh > 0;
          gain[u]    = gain_of(grads(ls.x), lh, grads(to_right.x - run.x), rh, parent);
          left_of[u] = ls;
        }
        // (a node without a candidate here is none of those that the thread has to report)
#pragma unroll
        for (int u = 0; u < kG; u++)
          if (wanted[u] && gain[u] > 0) {
            if (node[e0 + u] != cur) next_node(node[e0 + u]);
            offer(gain[u], e0 + u, left_of[u]);
          }
      }
    }
    // one slot for the node the thread begins with, one for the node it ends with (the same one, or none)
    if (first_node == kNone) {
      first_node = cur;
      first_gain = cur_gain;
      first_key  = cur_key;
      first_left = cur_left;
      cur_key    = 0;
    }
    const int own_node     = first_node;
    const unsigned own_key = first_key;
    const unsigned long long first_bits = static_cast<unsigned long long>(__double_as_longlong(first_gain));
    const unsigned long long cur_bits   = static_cast<unsigned long long>(__double_as_longlong(cur_gain));
    // where a whole wave lies in one node its lanes meet first
    const unsigned long long have = __ballot(first_key != 0 || cur_key != 0);
    bool alone = true;
    if (have != 0) {
      const int wave_node = __builtin_amdgcn_readlane(first_node, __builtin_ctzll(have));
      alone               = !__all(cur_key == 0 && (first_key == 0 || first_node == wave_node));
      if (!alone) {
        double top   = first_key != 0 ? first_gain : 0.0;
        unsigned key = first_key;
        wave_best_key(top, key);
        first_node = wave_node;
        first_gain = top;
        first_key  = lane == 0 ? key : 0u;
      }
    }
    const unsigned long long mine_bits = alone ? first_bits : static_cast<unsigned long long>(__double_as_longlong(first_gain));
    if (first_key != 0) atomicMax(&s_gain[first_node], mine_bits);
    if (cur_key != 0) atomicMax(&s_gain[cur], cur_bits);
    __syncthreads();
    if (first_key != 0 && mine_bits == s_gain[first_node]) atomicMax(&s_key[first_node], first_key);
    if (cur_key != 0 && cur_bits == s_gain[cur]) atomicMax(&s_key[cur], cur_key);
    __syncthreads();
    if constexpr (kLeft) {
      // (keys of different bins differ, but one lane can hold an equal key of a smaller gain only for another bin: none)
      if (own_key != 0 && own_key == s_key[own_node]) put_left(own_node, first_left);
      if (cur_key != 0 && cur_key == s_key[cur]) put_left(cur, cur_left);
    }
  } else {
    double gain[kE];
    unsigned dead = 0;
#pragma unroll
    for (int e = 0; e < kE; e++) gain[e] = 0.0;
    // The pairs of the next output, and what the nodes have of it, are on their way while this one's sums and gains are formed, and lie in the
    // LDS when they are asked for: gathered from the L2 place by place, with the nodes' sums behind the places' sums, they were two latencies
    // an output: 590 x 118 with 8 outputs, depth 9, 24.7 us a launch, and 20.5; 7000 x 300 with 2, depth 8, 96 and 83 (with
    // sums in 32 bits and plain quotients 17.1 and 65). kStaged: the nodes' sums, bases and terms of the gain, a thread each, those of one
    // output beside those of the next.
    I64Pair* const s_of_k    = reinterpret_cast<I64Pair*>(smem_raw + small_scan_use(a.N, a.n_nodes));  // [2][2][n_nodes]
    double* const s_parent_k = reinterpret_cast<double*>(s_of_k + 4 * a.n_nodes);                      // [2][n_nodes]
    const int64_t own_at     = static_cast<int64_t>(a.level_first + min(tid, a.n_nodes - 1)) * a.K;
    int2 q_next[kE];
    I64Pair ns_next{0, 0}, base_next{0, 0}, all_next{0, 0};
    const bool plain = plain_quotients(a.l1, inv_g, inv_h, reg);
    auto fetch = [&](int k) {
      all_next = st.node_sums[k];
#pragma unroll
      for (int u = 0; u < kE; u++) q_next[u] = st.qgh[min(tid + u * kT, a.N - 1) * a.K + k];
      if constexpr (kStaged) {
        ns_next   = st.node_sums[own_at + k];
        base_next = st.base[own_at + k];
      }
    };
    fetch(0);
    for (int k = 0; k < a.K; k++) {
      I64Pair* const ns_of = s_of_k + 2 * (k & 1) * a.n_nodes;
      I64Pair* const base_of = ns_of + a.n_nodes;
      double* const parent_of_k = s_parent_k + (k & 1) * a.n_nodes;
      // (nobody looks at the pairs of the output before any more: a barrier lies behind those looks)
#pragma unroll
      for (int u = 0; u < kE; u++)
        if (tid + u * kT < a.N) s_q[tid + u * kT] = q_next[u];
      if constexpr (kStaged) {
        if (tid < a.n_nodes) {
          ns_of[tid]       = ns_next;
          base_of[tid]     = base_next;
          parent_of_k[tid] = leaf_gain(static_cast<double>(ns_next.grad) * inv_g, static_cast<double>(ns_next.hess) * inv_h, a.l1, reg);
        }
      }
      // (sums in their lower 32 bits, as with one output)
      const int64_t most   = (int64_t(1) << 31) + a.N + 1024;
      const uint32_t down_g = static_cast<uint32_t>((most - all_next.grad) / 2 + 1), down_h = static_cast<uint32_t>((most - all_next.hess) / 2 + 1);
      const double from_g = static_cast<double>(down_g), from_h = static_cast<double>(down_h);
      if (k + 1 < a.K) fetch(k + 1);
      __syncthreads();
      int2 q[kE];
      uint2 sum = make_uint2(0, 0);
#pragma unroll
      for (int e = 0; e < kE; e++) {
        q[e] = i0 + e < a.N ? s_q[entry[e] & 0xffff] : make_int2(0, 0);
        sum.x += static_cast<uint32_t>(q[e].x);
        sum.y += static_cast<uint32_t>(q[e].y);
      }
      const uint32_t ig = wave_inclusive_sum32(sum.x);
      const uint32_t ih = wave_inclusive_sum32(sum.y);
      uint2* const s_tot = reinterpret_cast<uint2*>(s_pair[k & 1]);
      if (lane == 63) s_tot[wave] = make_uint2(ig, ih);
      __syncthreads();
      uint2 before = make_uint2(ig - sum.x, ih - sum.y);
      for (int w = 0; w < kT / 64; w++) {
        before.x += w < wave ? s_tot[w].x : 0;
        before.y += w < wave ? s_tot[w].y : 0;
      }
      auto offer = [&](int e, int j, auto plains) {
        I64Pair ns, base;
        double parent;
        if constexpr (kStaged) {
          ns     = ns_of[j];
          base   = base_of[j];
          parent = parent_of_k[j];
        } else {
          const int64_t at = static_cast<int64_t>(a.level_first + j) * a.K + k;
          ns     = st.node_sums[at];
          base   = st.base[at];
          parent = leaf_gain_select(static_cast<double>(ns.grad) * inv_g, static_cast<double>(ns.hess) * inv_h, a.l1, reg);
        }
        auto quotient = [&](double grad, double hess) {
          if constexpr (decltype(plains)::value)
            return quotient_plain(grad * grad, hess + reg);
          else
            return leaf_gain_select(grad, hess, a.l1, reg);
        };
        const uint32_t g = before.x - static_cast<uint32_t>(base.grad), h = before.y - static_cast<uint32_t>(base.hess);
        const double lg = static_cast<double>(g + down_g) - from_g, rg = static_cast<double>(static_cast<uint32_t>(ns.grad) - g + down_g) - from_g;
        const double lh = static_cast<double>(h + down_h) - from_h, rh = static_cast<double>(static_cast<uint32_t>(ns.hess) - h + down_h) - from_h;
        // build_tree.cu:727-730: one output without a valid split on this bin voids the bin
        dead |= lh <= 0 || rh <= 0 ? 1u << e : 0u;
        gain[e] += (0.5 * (quotient(lg * inv_g, lh * inv_h) + quotient(rg * inv_g, rh * inv_h) - parent)) - a.min_split_gain;
      };
      // a few waves: the places' quotients side by side, without branches (a place whose bin does not end there has no say below);
      // sixteen of them hide each other's chains, and only the places that have a say are worth the time
      auto offer_all = [&](auto plains) {
#pragma unroll
        for (int e = 0; e < kE; e++) {
          before.x += static_cast<uint32_t>(q[e].x);
          before.y += static_cast<uint32_t>(q[e].y);
          if constexpr (kT < 1024)
            offer(e, node[e] != kNone ? node[e] : 0, plains);
          else if (((ends & ~dead) >> e) & 1u)
            offer(e, node[e], plains);
        }
      };
      if (plain)
        offer_all(std::true_type{});
      else
        offer_all(std::false_type{});
    }
    ends &= ~dead;
    // best gain per node: a thread's runs of one node first, then, where a whole wave lies in one
    // node, the wave
    {
      int run_node = kNone, runs = 0;
      double run_gain = 0.0;
#pragma unroll
      for (int e = 0; e < kE; e++) {
        const bool has = ((ends >> e) & 1u) != 0 && gain[e] > 0;
        if (has) {
          if (node[e] != run_node) {
            if (runs > 0) atomicMax(&s_gain[run_node], static_cast<unsigned long long>(__double_as_longlong(run_gain)));
            run_node = node[e];
            run_gain = gain[e];
            runs++;
          } else {
            run_gain = gain[e] > run_gain ? gain[e] : run_gain;
          }
        }
      }
      const unsigned long long have = __ballot(runs > 0);
      if (have != 0) {
        const int first_lane = __ffsll(have) - 1;
        const int wave_node  = __shfl(run_node, first_lane, 64);
        if (__all(runs == 0 || run_node == wave_node)) {
          for (int off = 32; off >= 1; off >>= 1) {
            const double o = __shfl_xor(run_gain, off, 64);
            run_gain       = o > run_gain ? o : run_gain;
          }
          if (lane == 0) atomicMax(&s_gain[wave_node], static_cast<unsigned long long>(__double_as_longlong(run_gain)));
        } else if (runs > 0) {
          atomicMax(&s_gain[run_node], static_cast<unsigned long long>(__double_as_longlong(run_gain)));
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kE; e++) {
      if (((ends >> e) & 1u) != 0 && gain[e] > 0 &&
          static_cast<unsigned long long>(__double_as_longlong(gain[e])) == s_gain[node[e]]) {
        atomicMax(&s_key[node[e]], tie_key(rp, bin[e], bin[e + 1]));
      }
    }
    __syncthreads();
  }
  for (int j = tid; j < a.n_nodes; j += kT) {
    const unsigned key = s_key[j];  // (nodes without rows have none)
    SmallCand c{0.0, 0u, 0};
    if (key != 0) {
      c.gain = __longlong_as_double(static_cast<long long>(s_gain[j]));
      c.rel  = 2047 - static_cast<int>((key - 1u) & 2047u);
      c.key  = tie_key_of_bin(rp + c.rel);
    }
    out[static_cast<int64_t>(j) * a.F] = c;
  }
  if constexpr (kDecides) write_outputs();
}

// Split of one node, its outputs, its children and the side of each of its rows.
template <int kT>
__global__ void __launch_bounds__(kT)
  small_apply_kernel(SmallTreeState st, LevelArgs a, uint16_t* node_of_pos)
{
  __shared__ double s_best[kT / 64];
  __shared__ int4 s_pick[kT / 64];
  __shared__ int s_cnt[kT / 64];
  __shared__ I64Pair s_sum[2][kT / 64];
  const int j    = blockIdx.x;
  const int node = a.level_first + j;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int live      = st.live[a.depth];
  const int2 seg      = st.seg[node];
  // what only the last lines need is asked for here
  const double inv_g = st.scales[2], inv_h = st.scales[3];
  const I64Pair ns0 = st.node_sums[static_cast<int64_t>(node) * a.K], base0 = st.base[static_cast<int64_t>(node) * a.K];
  const int s0 = seg.x, n = seg.y;
  if (live == 0 || n == 0) return;
  const uint32_t* order = st.order[a.depth & 1] + s0;  // feature 0's
  // a thread's first row is asked for together with the candidates
  const uint32_t first_row = tid < n ? order[tid] & 0xffffu : 0u;
  auto row_at = [&](int i) { return i == tid ? first_row : order[i] & 0xffffu; };
  // the best candidate by (gain, key of the tie rule), without branches
  double best = 0.0;
  unsigned best_key = 0;
  int ft = 0, rel = 0;
  auto take = [&](double gain_o, unsigned key_o, int ft_o, int rel_o) {
    const bool better = gain_o > best || (gain_o == best && key_o > best_key);
    best     = better ? gain_o : best;
    best_key = better ? key_o : best_key;
    ft       = better ? ft_o : ft;
    rel      = better ? rel_o : rel;
  };
  const SmallCand* c = a.cand + static_cast<int64_t>(j) * a.F;
  for (int i = tid; i < a.F; i += kT) {
    const SmallCand o = c[i];
    take(o.gain, o.key, i, o.rel);
  }
  wave_best_split(best, best_key, ft, rel);
  if (kT > 64) {
    if (lane == 0) {
      s_best[wave] = best;
      s_pick[wave] = make_int4(static_cast<int>(best_key), ft, rel, 0);
    }
    __syncthreads();
    for (int w = 0; w < kT / 64; w++) {
      const int4 p = s_pick[w];
      take(s_best[w], static_cast<unsigned>(p.x), p.y, p.z);
    }
  }
  if (!(ns0.hess > 0 && best_key != 0 && best > 1e-5)) {
    for (int i = tid; i < n; i += kT) {
      node_of_pos[s0 + i] = kNone;
      if (a.row_leaf != nullptr) a.row_leaf[row_at(i)] = node;
    }
    return;
  }
  const int lc = left_child(node), rc = right_child(node);
  const uint16_t* bins = st.bins + static_cast<int64_t>(ft) * st.pitch;
  const double value   = st.proposals[static_cast<int64_t>(ft) * a.S + rel];
  int nl = 0;
  I64Pair sum{0, 0};
  for (int i = tid; i < n; i += kT) {
    const int r     = static_cast<int>(row_at(i));
    const int2 q    = st.qgh[r * a.K];  // (asked for beside the bin)
    const bool left = bins[r] <= rel;
    if (!a.last) st.code[r] = left ? 1 : 2;
    if (a.last && a.row_leaf != nullptr) a.row_leaf[r] = left ? lc : rc;
    if (left) {
      nl++;
      sum.grad += q.x;
      sum.hess += q.y;
    }
  }
  for (int k = 0;;) {
    const int64_t ig = wave_inclusive_sum(sum.grad), ih = wave_inclusive_sum(sum.hess);
    if (lane == 63) s_sum[k & 1][wave] = I64Pair{ig, ih};
    if (k == 0) {
      const int c = static_cast<int>(wave_inclusive_sum32(static_cast<uint32_t>(nl)));
      if (lane == 63) s_cnt[wave] = c;
    }
    __syncthreads();
    if (tid < 2) {
      // a child each, the left one first
      I64Pair ls{0, 0};
      for (int w = 0; w < kT / 64; w++) {
        ls.grad += s_sum[k & 1][w].grad;
        ls.hess += s_sum[k & 1][w].hess;
      }
      const int64_t at = static_cast<int64_t>(node) * a.K + k, to = static_cast<int64_t>(tid == 0 ? lc : rc) * a.K + k;
      const I64Pair ns = k == 0 ? ns0 : st.node_sums[at], base = k == 0 ? base0 : st.base[at];
      const I64Pair own{tid == 0 ? ls.grad : ns.grad - ls.grad, tid == 0 ? ls.hess : ns.hess - ls.hess};
      st.node_sums[to] = own;
      st.base[to]      = I64Pair{base.grad + (tid == 0 ? 0 : ls.grad), base.hess + (tid == 0 ? 0 : ls.hess)};
      const double g = static_cast<double>(own.grad) * inv_g, h = static_cast<double>(own.hess) * inv_h;
      a.leaf[to]    = calculate_leaf_value(g, h, a.l1, a.l2);
      a.hessian[to] = h;
    }
    if (++k == a.K) break;
    sum = I64Pair{0, 0};
    for (int i = tid; i < n; i += kT) {
      const int r = static_cast<int>(row_at(i));
      if (bins[r] <= rel) {
        const int2 q = st.qgh[r * a.K + k];
        sum.grad += q.x;
        sum.hess += q.y;
      }
    }
  }
  int lefts = 0;
  for (int w = 0; w < kT / 64; w++) lefts += s_cnt[w];
  if (tid == 0) {
    a.feature[node] = ft;
    a.split[node]   = value;
    a.gain[node]    = best;
    st.seg[lc]    = make_int2(s0, lefts);
    st.seg[rc]    = make_int2(s0 + lefts, n - lefts);
    st.live[a.depth + 1] = 1;
  }
  if (!a.last)
    for (int i = tid; i < n; i += kT) node_of_pos[s0 + i] = static_cast<uint16_t>(2 * j + (i < lefts ? 0 : 1));
}

// ---------------------------------------------------------------- all levels in one launch

constexpr int kLevelsMaxDepth = 10;
constexpr int kLevelsPolls    = 400;   // looks (about 0.7 us apart) at what the others find before a workgroup takes a feature over

thread_local int levels_polls = kLevelsPolls;

struct LevelsArgs {
  int N, F, S, max_depth;
  int lanes_log;  // lanes per node where a level is decided, log2: at least F
  bool all_bins;  // the bins of all features lie in the LDS
  int polls;
  double* leaf;
  int32_t* feature;
  double* split;
  double* gain;
  double* hessian;
  int32_t* row_leaf;
  unsigned long long* n_bins;  // pinned host memory: the number of all bins (see DeviceAnswer)
  uint32_t tag;
  const uint8_t* feature_set;
  double l1, l2, min_split_gain;
};

__host__ __device__ constexpr size_t small_levels_use(int64_t N, int max_depth)
{
  return static_cast<size_t>((N + 1) / 2 * 2 * 8 + small_scan_order(N) * 4 + (int64_t(1) << (max_depth - 1)) * 100 + 15) / 16 * 16;
}

__device__ __forceinline__ unsigned long long agent_load(const unsigned long long* p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void agent_store(unsigned long long* p, unsigned long long v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// small_scan_kernel and the decisions between its levels for trees of one output, up to 64 features and 4096 rows: a workgroup keeps its
// feature's order in registers and the nodes in the LDS from level to level, and the workgroups tell each other what they found through memory:
// per node with rows and feature the gain, the place among equal gains and what lies left of the split, a word each that no launch
// has written before (the prologue leaves kNotFound in all of them), so that a word is its own signal.
// st.found: [node][gain, key and bin, left sums][F]; st.sync[f]: feature f has a workgroup.
// No workgroup waits for one that may not run: a feature belongs to the workgroup that takes it first, which is its own unless that has not started
// when another one has looked `polls` times for what it finds in the root; that one then takes the feature over. A workgroup with several features keeps their orders in memory.
template <int kT, int kE>
__global__ void __launch_bounds__(kT) small_levels_kernel(SmallTreeState st, LevelsArgs a)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int most = 1 << (a.max_depth - 1);  // nodes of a level
  int2* const s_q                  = reinterpret_cast<int2*>(smem_raw);                              // [N]
  uint32_t* const s_order          = reinterpret_cast<uint32_t*>(s_q + (a.N + 1) / 2 * 2);          // [small_scan_order(N)]
  unsigned long long* const s_gain = reinterpret_cast<unsigned long long*>(s_order + small_scan_order(a.N));  // [most], as the others
  double* const s_parent           = reinterpret_cast<double*>(s_gain + most);
  double* const s_best             = s_parent + most;
  uint2* const s_sums              = reinterpret_cast<uint2*>(s_best + most);   // [2][most] lower halves, as s_base and s_left
  uint2* const s_bases             = s_sums + 2 * most;                          // [2][most]
  int2* const s_segs               = reinterpret_cast<int2*>(s_bases + 2 * most);  // [2][most]
  uint2* const s_left              = reinterpret_cast<uint2*>(s_segs + 2 * most);
  int2* const s_split              = reinterpret_cast<int2*>(s_left + most);
  unsigned* const s_key            = reinterpret_cast<unsigned*>(s_split + most);
  int* const s_left_before         = reinterpret_cast<int*>(s_key + most);
  int* const s_left_behind         = s_left_before + most;
  uint16_t* const s_bins           = reinterpret_cast<uint16_t*>(smem_raw + small_levels_use(a.N, a.max_depth));  // all_bins: [F][pitch]
  __shared__ uint2 s_wave_sums[kT / 64];
  __shared__ int s_wave[kT / 64];
  __shared__ unsigned s_taken;
  __shared__ unsigned long long s_over;
  __shared__ int s_splits;  // the last level with a split, counted from 1
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i0   = tid * kE;
  const int pitch = static_cast<int>(st.pitch);
  // features that are candidates, those with a workgroup (feature 0's writes the outputs), and the first bin of each
  const unsigned long long usable = __ballot(lane < a.F && (a.feature_set == nullptr || a.feature_set[min(lane, a.F - 1)] != 0));
  const unsigned long long parts  = usable | 1ull;
  const int n_parts               = __popcll(parts);
  const int bins_here             = lane < a.F ? st.counts[lane] : 0;
  if (static_cast<int>(blockIdx.x) >= n_parts) return;
  unsigned long long behind = parts;
  for (int i = 0; i < static_cast<int>(blockIdx.x); i++) behind &= behind - 1;
  const int f_first = __builtin_ctzll(behind);
  if (tid == 0) s_taken = __hip_atomic_exchange(&st.sync[f_first], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int live     = st.live[0];
  const double inv_g = st.scales[2], inv_h = st.scales[3];
  const I64Pair all  = st.node_sums[0];
  const double reg   = 1e-5 > a.l2 ? 1e-5 : a.l2;
  uint32_t entry[kE];
  load_u32<kE>(st.order[0] + static_cast<int64_t>(f_first) * pitch + min(i0, pitch - kE), entry);
  {
    int2 pair[kE];
#pragma unroll
    for (int u = 0; u < kE; u++) pair[u] = st.qgh[min(tid + u * kT, a.N - 1)];
    if (a.all_bins)
      copy_ahead<kT, 4>(a.F * (pitch / 8), [&](int i) { return reinterpret_cast<const uint4*>(st.bins)[i]; },
                        [&](int i, const uint4& v) { reinterpret_cast<uint4*>(s_bins)[i] = v; });
#pragma unroll
    for (int u = 0; u < kE; u++)
      if (tid + u * kT < a.N) s_q[tid + u * kT] = pair[u];
  }
  const int bins_before = static_cast<int>(wave_inclusive_sum32(static_cast<uint32_t>(bins_here))) - bins_here;
  if (f_first == 0 && tid == 0)
    __hip_atomic_store(a.n_bins,
                       (static_cast<unsigned long long>(a.tag) << 32) |
                         static_cast<unsigned>(__builtin_amdgcn_readlane(bins_before + bins_here, 63)),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (live == 0) return;  // data for the other builder
  // sums are formed in their lower halves, see small_scan_kernel
  const int64_t range  = (int64_t(1) << 31) + a.N + 1024;
  const uint32_t down_g = static_cast<uint32_t>((range - all.grad) / 2 + 1), down_h = static_cast<uint32_t>((range - all.hess) / 2 + 1);
  const double from_g = static_cast<double>(down_g), from_h = static_cast<double>(down_h);
  auto grads  = [&](uint32_t v) { return static_cast<double>(v) - from_g; };  // of a sum with `down` added
  auto hesses = [&](uint32_t v) { return static_cast<double>(v) - from_h; };
  if (tid == 0) {
    s_splits    = 0;
    s_over      = 0;
    s_sums[0]   = make_uint2(static_cast<uint32_t>(all.grad), static_cast<uint32_t>(all.hess));
    s_bases[0]  = make_uint2(0, 0);
    s_segs[0]   = make_int2(0, a.N);
    s_parent[0] = leaf_gain(static_cast<double>(all.grad) * inv_g, static_cast<double>(all.hess) * inv_h, a.l1, reg);
  }
  const bool plain = plain_quotients(a.l1, inv_g, inv_h, reg);
  auto term_of = [&](double grad, double hess) { return plain ? quotient_plain(grad * grad, hess + reg) : leaf_gain(grad, hess, a.l1, reg); };
  auto gain_of = [&](double lg, double lh, double rg, double rh, double parent) {
    lg *= inv_g, rg *= inv_g, lh *= inv_h, rh *= inv_h;
    if (plain) return 0.0 + ((0.5 * (quotient_plain(lg * lg, lh + reg) + quotient_plain(rg * rg, rh + reg) - parent)) - a.min_split_gain);
    return 0.0 + ((0.5 * (leaf_gain(lg, lh, a.l1, reg) + leaf_gain(rg, rh, a.l1, reg) - parent)) - a.min_split_gain);
  };
  // (the writer) node `at` has split: its outputs and its children's
  auto write_split = [&](int at, const int2& s, double best, const uint2& ls, const uint2& rs) {
    const int to       = 2 * at + 1;
    const double value = st.proposals[static_cast<int64_t>(s.x) * a.S + s.y];
    const double lg = grads(ls.x + down_g) * inv_g, lh = hesses(ls.y + down_h) * inv_h;
    const double rg = grads(rs.x + down_g) * inv_g, rh = hesses(rs.y + down_h) * inv_h;
    a.feature[at]     = s.x;
    a.gain[at]        = best;
    a.leaf[to]        = calculate_leaf_value(lg, lh, a.l1, a.l2);
    a.leaf[to + 1]    = calculate_leaf_value(rg, rh, a.l1, a.l2);
    a.hessian[to]     = lh;
    a.hessian[to + 1] = rh;
    a.split[at]       = value;
  };
  int node[kE], child[kE], node_next, child_next;
#pragma unroll
  for (int e = 0; e < kE; e++) node[e] = child[e] = i0 + e < a.N ? 0 : kNone;
  node_next = child_next = i0 + kE < a.N ? 0 : kNone;
  __syncthreads();
  if (s_taken != 0) return;
  unsigned long long owned = 1ull << f_first, todo = owned;
  bool writes       = f_first == 0;
  bool first_here   = true;  // the first feature of the level
  for (int d = 0;;) {
    const int n_nodes = 1 << d, n_above = n_nodes / 2, above_first = n_above - 1;
    const int cur = (d & 1) * most, above = most - cur;  // this level's half of the nodes' sums, and the other one
    const bool single = (owned & (owned - 1)) == 0;
    const int f       = __builtin_ctzll(todo);
    todo &= todo - 1;
    const int rp = __builtin_amdgcn_readlane(bins_before, f);
    if (!single || (d == 0 && !first_here))
      load_u32<kE>(st.order[d == 0 ? 0 : (d - 1) & 1] + static_cast<int64_t>(f) * pitch + min(i0, pitch - kE), entry);
    for (int j = tid; j < n_nodes; j += kT) {
      s_gain[j] = 0;
      s_key[j]  = 0;
    }
    if (d > 0) {
      // the feature's order of this level: a stable partition inside every node that has split
      unsigned left = 0, goes_on = 0;
      int2 sp[kE], at[kE];
      int b[kE];
#pragma unroll
      for (int e = 0; e < kE; e++) {
        // (no branches around the looks into the LDS: behind one, each is waited for before the next is asked for)
        const int2 s = s_split[node[e] != kNone ? node[e] : 0];
        sp[e]        = make_int2(node[e] != kNone ? s.x : -1, s.y);
        at[e]        = s_segs[above + (node[e] != kNone ? node[e] : 0)];
      }
      auto bin_at = [&](int e) { return max(sp[e].x, 0) * pitch + min(static_cast<int>(entry[e] & 0xffff), a.N - 1); };
      if (a.all_bins) {
#pragma unroll
        for (int e = 0; e < kE; e++) b[e] = s_bins[bin_at(e)];
      } else {
#pragma unroll
        for (int e = 0; e < kE; e++) b[e] = st.bins[bin_at(e)];
      }
      if (writes && first_here && a.row_leaf != nullptr) {
#pragma unroll
        for (int e = 0; e < kE; e++)
          if (node[e] != kNone && sp[e].x < 0) a.row_leaf[entry[e] & 0xffff] = above_first + node[e];
      }
#pragma unroll
      for (int e = 0; e < kE; e++) {
        goes_on |= sp[e].x >= 0 ? 1u << e : 0u;
        left |= sp[e].x >= 0 && b[e] <= sp[e].y ? 1u << e : 0u;
      }
      const int before = block_exclusive_sum32<kT>(__popc(left), s_wave);
#pragma unroll
      for (int e = 0; e < kE; e++)
        if ((goes_on >> e) & 1u) {
          if (at[e].x == i0 + e) s_left_before[node[e]] = before + __popc(left & ((1u << e) - 1u));
          if (at[e].x + at[e].y - 1 == i0 + e) s_left_behind[node[e]] = before + __popc(left & ((2u << e) - 1u));
        }
      const int next          = node_next != kNone ? node_next : 0;
      const bool next_goes_on = node_next != kNone && s_split[next].x >= 0;
      const int2 next_at      = s_segs[above + next];
      const int mine          = min(tid, n_above - 1);
      const bool splits       = s_split[mine].x >= 0;
      const int2 mine_at      = s_segs[above + mine];
      __syncthreads();
      int first[kE], lefts[kE];
#pragma unroll
      for (int e = 0; e < kE; e++) {
        const int j = node[e] != kNone ? node[e] : 0;
        first[e]    = s_left_before[j];
        lefts[e]    = s_left_behind[j] - first[e];
      }
      const int next_lefts = s_left_behind[next] - s_left_before[next], mine_lefts = s_left_behind[mine] - s_left_before[mine];
#pragma unroll
      for (int e = 0; e < kE; e++) {
        const int i = i0 + e;
        const int l = before + __popc(left & ((1u << e) - 1u)) - first[e];
        const bool goes = ((goes_on >> e) & 1u) != 0;
        const int to    = !goes ? i : (left >> e) & 1u ? at[e].x + l : i + lefts[e] - l;
        child[e]        = goes ? 2 * node[e] + (i - at[e].x < lefts[e] ? 0 : 1) : kNone;
        if (i < a.N) s_order[to] = entry[e];
      }
      child_next = next_goes_on ? 2 * node_next + (i0 + kE - next_at.x < next_lefts ? 0 : 1) : kNone;
      if (tid < n_above) {
        s_segs[cur + 2 * tid]     = make_int2(mine_at.x, splits ? mine_lefts : 0);
        s_segs[cur + 2 * tid + 1] = make_int2(mine_at.x + (splits ? mine_lefts : 0), splits ? mine_at.y - mine_lefts : 0);
      }
      __syncthreads();
      if (i0 < a.N) load_u32<kE>(s_order + i0, entry);
      if (!single && i0 < a.N) store_u32<kE>(st.order[d & 1] + static_cast<int64_t>(f) * pitch + i0, entry);
    } else {
      // the neighbour's first bin is looked up below
      if (i0 < a.N) s_order[i0] = entry[0];
      __syncthreads();
    }
    unsigned long long* const found = st.found + static_cast<int64_t>(n_nodes - 1) * 3 * a.F + f;  // node j: found[(3 * j + word) * F]
    // (the writer) what the level above has to write, taken before this level's splits lie there
    int2 was_split = make_int2(-1, 0);
    double was_best = 0.0;
    uint2 was_left = make_uint2(0, 0), was_right = make_uint2(0, 0);
    if (writes && first_here && tid < n_above) {
      was_split = s_split[tid];
      was_best  = s_best[tid];
      was_left  = s_sums[cur + 2 * tid];
      was_right = s_sums[cur + 2 * tid + 1];
    }
    if ((usable >> f & 1) != 0) {
      // occupied bins, running sums and gains, the best split per node: as small_scan_kernel
      int bin[kE + 1];
#pragma unroll
      for (int e = 0; e < kE; e++) bin[e] = static_cast<int>(entry[e] >> 16);
      bin[kE] = i0 + kE < a.N ? static_cast<int>(s_order[i0 + kE] >> 16) : 0;
      unsigned ends = 0;
#pragma unroll
      for (int e = 0; e < kE; e++) {
        const int nn = e + 1 < kE ? child[e + 1] : child_next;
        if (child[e] != kNone && nn == child[e] && bin[e + 1] != bin[e]) ends |= 1u << e;
      }
      int2 q[kE];
      uint2 sum = make_uint2(0, 0);
#pragma unroll
      for (int e = 0; e < kE; e++) {
        q[e] = i0 + e < a.N ? s_q[entry[e] & 0xffff] : make_int2(0, 0);
        sum.x += static_cast<uint32_t>(q[e].x);
        sum.y += static_cast<uint32_t>(q[e].y);
      }
      const uint32_t ig = wave_inclusive_sum32(sum.x), ih = wave_inclusive_sum32(sum.y);
      if (lane == 63) s_wave_sums[wave] = make_uint2(ig, ih);
      __syncthreads();
      uint2 run = make_uint2(ig - sum.x, ih - sum.y);
#pragma unroll
      for (int w = 0; w < kT / 64; w++) {
        run.x += w < wave ? s_wave_sums[w].x : 0;
        run.y += w < wave ? s_wave_sums[w].y : 0;
      }
      int first_node = kNone, own = kNone;
      double first_gain = 0.0, own_gain = 0.0;
      unsigned first_key = 0, own_key = 0;
      uint2 first_left = make_uint2(0, 0), own_left = make_uint2(0, 0);  // with `down` added
      auto put_left = [&](int j, const uint2& left) {
        agent_store(found + static_cast<int64_t>(3 * j + 2) * a.F, static_cast<unsigned long long>(left.x) << 32 | left.y);
      };
      double gain[kE];
      bool wanted[kE];
      uint2 left_of[kE];
#pragma unroll
      for (int e = 0; e < kE; e++) {
        run.x += static_cast<uint32_t>(q[e].x);
        run.y += static_cast<uint32_t>(q[e].y);
        const int j       = cur + (child[e] != kNone ? child[e] : 0);
        const uint2 total = s_sums[j], base = s_bases[j];
        const double parent = s_parent[j - cur];
        const uint2 ls  = make_uint2(run.x + down_g - base.x, run.y + down_h - base.y);
        const uint2 rs  = make_uint2(total.x + base.x + down_g - run.x, total.y + base.y + down_h - run.y);
        const double lh = hesses(ls.y), rh = hesses(rs.y);
        wanted[e]  = ((ends >> e) & 1u) != 0 && lh > 0 && rh > 0;
        gain[e]    = gain_of(grads(ls.x), lh, grads(rs.x), rh, parent);
        left_of[e] = ls;
      }
      // (a node without a candidate here is none of those that the thread has to report)
#pragma unroll
      for (int e = 0; e < kE; e++)
        if (wanted[e] && gain[e] > 0) {
          if (child[e] != own) {
            if (first_node == kNone) {
              first_node = own;  // (kNone again while there was none before)
              first_gain = own_gain;
              first_key  = own_key;
              first_left = own_left;
            } else if (own_key != 0) {
              s_gain[own] = static_cast<unsigned long long>(__double_as_longlong(own_gain));
              s_key[own]  = own_key;
              put_left(own, own_left);
            }
            own      = child[e];
            own_gain = 0.0;
            own_key  = 0;
          }
          if (gain[e] >= own_gain) {
            const unsigned key = tie_key(rp, bin[e], bin[e + 1]);
            const bool better  = gain[e] > own_gain || key > own_key;
            own_left.x         = better ? left_of[e].x : own_left.x;
            own_left.y         = better ? left_of[e].y : own_left.y;
            own_key            = gain[e] > own_gain ? key : max(own_key, key);
            own_gain           = gain[e];
          }
        }
      // one slot for the node the thread begins with, one for the node it ends with (the same one, or none)
      if (first_node == kNone) {
        first_node = own;
        first_gain = own_gain;
        first_key  = own_key;
        first_left = own_left;
        own_key    = 0;
      }
      const int begins_in      = first_node;
      const unsigned begin_key = first_key;
      const unsigned long long first_bits = static_cast<unsigned long long>(__double_as_longlong(first_gain));
      const unsigned long long own_bits   = static_cast<unsigned long long>(__double_as_longlong(own_gain));
      // where a whole wave lies in one node its lanes meet first
      const unsigned long long have = __ballot(first_key != 0 || own_key != 0);
      bool alone = true;
      if (have != 0) {
        const int wave_node = __builtin_amdgcn_readlane(first_node, __builtin_ctzll(have));
        alone               = !__all(own_key == 0 && (first_key == 0 || first_node == wave_node));
        if (!alone) {
          double top   = first_key != 0 ? first_gain : 0.0;
          unsigned key = first_key;
          wave_best_key(top, key);
          first_node = wave_node;
          first_gain = top;
          first_key  = lane == 0 ? key : 0u;
        }
      }
      const unsigned long long mine_bits = alone ? first_bits : static_cast<unsigned long long>(__double_as_longlong(first_gain));
      if (first_key != 0) atomicMax(&s_gain[first_node], mine_bits);
      if (own_key != 0) atomicMax(&s_gain[own], own_bits);
      __syncthreads();
      if (first_key != 0 && mine_bits == s_gain[first_node]) atomicMax(&s_key[first_node], first_key);
      if (own_key != 0 && own_bits == s_gain[own]) atomicMax(&s_key[own], own_key);
      __syncthreads();
      // (keys of different bins differ, but one lane can hold an equal key of a smaller gain only for another bin: none)
      if (begin_key != 0 && begin_key == s_key[begins_in]) put_left(begins_in, first_left);
      if (own_key != 0 && own_key == s_key[own]) put_left(own, own_left);
      for (int j = tid; j < n_nodes; j += kT) {
        if (s_segs[cur + j].y == 0) continue;  // nobody asks
        const unsigned key = s_key[j];
        const int rel      = 2047 - static_cast<int>((key - 1u) & 2047u);
        unsigned long long* const to = found + static_cast<int64_t>(3 * j) * a.F;
        agent_store(to, key != 0 ? s_gain[j] : 0ull);
        agent_store(to + a.F, key != 0 ? static_cast<unsigned long long>(tie_key_of_bin(rp + rel)) << 32 | static_cast<unsigned>(rel) : 0ull);
        if (key == 0) agent_store(to + 2 * a.F, 0ull);
      }
    } else {
      __syncthreads();  // (as the feature's sums do: the splits of the level above are no longer asked for)
    }
    if (was_split.x >= 0) write_split(above_first + tid, was_split, was_best, was_left, was_right);
    first_here = false;
    if (todo != 0 || !single) __syncthreads();  // (the next feature's places)
    if (todo != 0) continue;
    if (d + 1 == a.max_depth && !writes) return;
    // the splits of the level's nodes: 2^lanes_log lanes a node, a feature each
    const int up = cur, down = above;
    const int sub = tid & ((1 << a.lanes_log) - 1), turn = kT >> a.lanes_log;
    const bool asks = sub < a.F && (usable >> min(sub, 63) & 1) != 0;
    constexpr int kTurns = 2;
    for (int j0 = tid >> a.lanes_log; j0 - (tid >> a.lanes_log) < n_nodes; j0 += kTurns * turn) {
      unsigned long long g_of[kTurns], k_of[kTurns], l_of[kTurns];
      bool here[kTurns];
#pragma unroll
      for (int u = 0; u < kTurns; u++) here[u] = asks && j0 + u * turn < n_nodes && s_segs[up + min(j0 + u * turn, n_nodes - 1)].y > 0;
      bool any = false;
#pragma unroll
      for (int u = 0; u < kTurns; u++) {
        any |= here[u];
        g_of[u] = k_of[u] = l_of[u] = 0;
      }
      for (int polls = 0; __any(any);) {
#pragma unroll
        for (int u = 0; u < kTurns; u++) {
          const unsigned long long* const at = st.found + static_cast<int64_t>(3 * (n_nodes - 1 + min(j0 + u * turn, n_nodes - 1))) * a.F + min(sub, a.F - 1);
          g_of[u] = agent_load(at);
          k_of[u] = agent_load(at + a.F);
          l_of[u] = agent_load(at + 2 * a.F);
        }
        bool waits = false;
#pragma unroll
        for (int u = 0; u < kTurns; u++) waits |= here[u] && (g_of[u] == kNotFound || k_of[u] == kNotFound || l_of[u] == kNotFound);
        if (!__any(waits)) break;
        if (d > 0 || ++polls <= a.polls) continue;
        // a feature of the root without a workgroup, or with one that is on its way
        polls = 0;
        const unsigned long long alone = __ballot(waits && __hip_atomic_load(&st.sync[sub], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0);
        const bool takes = alone != 0 && lane == static_cast<int>(__builtin_ctzll(alone)) &&
                           __hip_atomic_exchange(&st.sync[sub], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
        if (__any(takes)) {
          if (takes) s_over = 1ull << sub;
          break;
        }
      }
#pragma unroll
      for (int u = 0; u < kTurns; u++) {
        // gains are not negative: their bits compare as whole numbers, upper halves first
        const int j           = j0 + u * turn;
        const unsigned own_hi = here[u] ? static_cast<unsigned>(g_of[u] >> 32) : 0u, own_lo = here[u] ? static_cast<unsigned>(g_of[u]) : 0u;
        const unsigned own_key = here[u] ? static_cast<unsigned>(k_of[u] >> 32) : 0u;
        const unsigned hi  = group_max_u32(own_hi, a.lanes_log);
        const unsigned lo  = group_max_u32(own_hi == hi ? own_lo : 0u, a.lanes_log);
        const unsigned key = group_max_u32(own_hi == hi && own_lo == lo ? own_key : 0u, a.lanes_log);
        const double best  = __longlong_as_double(static_cast<int64_t>(static_cast<uint64_t>(hi) << 32 | lo));
        const bool splits  = key != 0 && best > 1e-5;
        if (j < n_nodes) {
          if (!splits && sub == 0) s_split[j] = make_int2(-1, 0);
          if (splits && here[u] && own_hi == hi && own_lo == lo && own_key == key) {  // (keys of different candidates differ: one lane)
            s_splits   = d + 1;
            s_split[j] = make_int2(sub, static_cast<int>(k_of[u] & 0xffffffffull));
            s_best[j]  = best;
            s_left[j]  = make_uint2(static_cast<uint32_t>(l_of[u] >> 32) - down_g, static_cast<uint32_t>(l_of[u]) - down_h);
          }
        }
      }
    }
    __syncthreads();
    if (d == 0 && s_over != 0) {
      // features that this workgroup has taken over
      todo = s_over;
      owned |= todo;
      writes |= (todo & 1) != 0;
      __syncthreads();
      if (tid == 0) {
        s_over   = 0;
        s_splits = 0;
      }
      continue;
    }
    d++;
    todo       = owned;
    first_here = true;
#pragma unroll
    for (int e = 0; e < kE; e++) node[e] = child[e];
    node_next = child_next;
    const int n_up = n_nodes, up_first = n_nodes - 1;
    const bool ends = d == a.max_depth || s_splits != d;
    if (!ends && tid < 2 * n_up) {
      // (a thread for each child; without a split they have no rows and nobody asks for them)
      const int j = tid >> 1, side = tid & 1;
      const bool splits = s_split[j].x >= 0;
      const uint2 total = s_sums[up + j], base = s_bases[up + j], ls = splits ? s_left[j] : make_uint2(0, 0);
      const uint2 own   = side == 0 || !splits ? ls : make_uint2(total.x - ls.x, total.y - ls.y);
      s_sums[down + tid]  = own;
      s_bases[down + tid] = side == 0 ? base : make_uint2(base.x + ls.x, base.y + ls.y);
      s_parent[tid]       = term_of(grads(own.x + down_g) * inv_g, hesses(own.y + down_h) * inv_h);
    }
    if (ends) {
      if (writes && tid < n_up && s_split[tid].x >= 0) {
        const uint2 total = s_sums[up + tid], ls = s_left[tid];
        write_split(up_first + tid, s_split[tid], s_best[tid], ls, make_uint2(total.x - ls.x, total.y - ls.y));
      }
      if (writes && a.row_leaf != nullptr) {
        if ((owned & (owned - 1)) != 0)
          load_u32<kE>(st.order[(d - 1) & 1] + min(i0, pitch - kE), entry);  // (feature 0's)
#pragma unroll
        for (int e = 0; e < kE; e++)
          if (node[e] != kNone) {
            const int2 s  = s_split[node[e]];
            const int row = static_cast<int>(entry[e] & 0xffff), at = up_first + node[e];
            a.row_leaf[row] = s.x < 0 ? at : 2 * at + (st.bins[s.x * pitch + row] <= s.y ? 1 : 2);
          }
      }
      return;
    }
  }
}

// For the profiler: what the histograms of the level would be built from.
__global__ void __launch_bounds__(256) small_count_kernel(SmallTreeState st, LevelArgs a, LevelMeta* total)
{
  for (int j = threadIdx.x; j < a.n_nodes; j += 256) {
    const int node = a.level_first + j, n = st.seg[node].y;
    if (n == 0 || st.live[a.depth] == 0) continue;
    const bool built = compute_histogram_bin(node, st.node_sums, a.K, node != 0);
    atomicAdd(reinterpret_cast<unsigned long long*>(&total->instances), static_cast<unsigned long long>(n));
    if (built) {
      atomicAdd(reinterpret_cast<unsigned long long*>(&total->built_instances), static_cast<unsigned long long>(n));
      atomicAdd(reinterpret_cast<unsigned long long*>(&total->built_nodes), 1ULL);
    }
  }
}

template <int kT, int kE, bool kSingle, int kG, bool kStaged, bool kDecides, bool kLeft = kDecides>
int launch_small_scan_as(hipStream_t stream, const SmallTreeState& st, const LevelArgs& a, size_t lds)
{
  static std::atomic<bool> attr_set[kMaxDevices] = {};
  LBT_REQUIRE(small_scan_places(a.N) == kT * kE, "%d rows do not take a workgroup of %d places", a.N, kT * kE);
  LBT_TRY((allow_dynamic_lds(small_scan_kernel<kT, kE, kSingle, kG, kStaged, kDecides, kLeft>, kScanLds + 64, attr_set)));
  small_scan_kernel<kT, kE, kSingle, kG, kStaged, kDecides, kLeft><<<a.F, kT, lds, stream>>>(st, a);
  return LBT_OK;
}
size_t small_staged_use(int64_t N, int64_t n_nodes)
{
  return small_scan_use(N, n_nodes) + static_cast<size_t>(n_nodes) * (2 * sizeof(I64Pair) + sizeof(double) + sizeof(int2));
}
template <int kT, int kE>
int launch_small_scan(hipStream_t stream, const SmallTreeState& st, const LevelArgs& a, bool decides)
{
  constexpr int kG = kE == 8 ? 2 : 4;
  // a scan that decides has more to do per place: up to 1024 rows twice the threads with half the places each
  constexpr int kDT = kT == 256 ? 512 : kT, kDE = kT * kE / kDT;
  const size_t lds  = small_scan_use(a.N, a.n_nodes);
  const size_t more = small_staged_use(a.N, a.n_nodes);
  if constexpr (kE == 4) {
    if (decides) {
      LevelArgs b       = a;
      const size_t bins = static_cast<size_t>(a.F) * st.pitch * sizeof(uint16_t), all = more + small_decide_use(a.n_nodes);
      b.all_bins        = bins <= static_cast<size_t>(kDT) * 16 * decide_loads(kDT) && all + bins <= kScanLds;
      return launch_small_scan_as<kDT, kDE, true, kDE, true, true>(stream, st, b, all + (b.all_bins ? bins : 0));
    }
  }
  if (a.K > 1) {
    const size_t both = lds + static_cast<size_t>(a.n_nodes) * 2 * (2 * sizeof(I64Pair) + sizeof(double));
    // two outputs' nodes; no workgroup of the CU is given up for them (of 1024 threads with these registers there is one) where there are
    // more workgroups than CUs
    auto at_once = [](size_t bytes) { return std::min<size_t>(1024 / kT, 160 * 1024 / (bytes + 1024)); };
    if (a.n_nodes <= kT && both <= kScanLds && (a.F <= 256 || at_once(both) >= at_once(lds)))
      return launch_small_scan_as<kT, kE, false, 1, true, false>(stream, st, a, both);
    return launch_small_scan_as<kT, kE, false, 1, false, false>(stream, st, a, lds);
  }
  // staging must not cost a workgroup of the CU where there are more of them than CUs
  auto per_cu        = [](size_t bytes) { return static_cast<int>(std::min<size_t>(2048 / kT, 160 * 1024 / (bytes + 1024))); };
  const bool crowded = kT == 1024 && a.F > 256;
  if (more > kScanLds || (per_cu(more) < per_cu(lds) && a.F > 256 * per_cu(more)))
    return launch_small_scan_as<kT, kE, true, 1, false, false>(stream, st, a, lds);
  if (crowded) return launch_small_scan_as<kT, kE, true, 1, true, false>(stream, st, a, more);
  if constexpr (kE <= 4) {
    if (a.left != nullptr) return launch_small_scan_as<kT, kE, true, kG, true, false, true>(stream, st, a, more);
  }
  return launch_small_scan_as<kT, kE, true, kG, true, false>(stream, st, a, more);
}

template <int kT, int kE>
int launch_small_levels(hipStream_t stream, const SmallTreeState& st, const LevelsArgs& a, size_t lds)
{
  static std::atomic<bool> attr_set[kMaxDevices] = {};
  LBT_REQUIRE(a.N <= kT * kE && a.F <= kSmallDecideFeatures && a.max_depth <= kLevelsMaxDepth, "%d rows do not take a workgroup of %d places",
              a.N, kT * kE);
  LBT_TRY((allow_dynamic_lds(small_levels_kernel<kT, kE>, kScanLds, attr_set)));
  small_levels_kernel<kT, kE><<<a.F, kT, lds, stream>>>(st, a);
  return LBT_OK;
}

// Whether the scan of the level below level `depth` finds this level's splits for itself: one output, a lane for every
// feature and kDecidePasses of them for the nodes, a thread for every node, and the LDS for both levels' nodes.
bool next_scan_decides(const SmallTreeState& st, int64_t N, int F, int K, int depth, int max_depth)
{
  if (st.left[0] == nullptr || K > 1 || F > kSmallDecideFeatures || depth + 1 >= max_depth || N > kDecideRows) return false;
  const int threads = N <= 1024 ? 512 : small_scan_places(N) / 4;
  int lanes = 1 << kDecideLanes;
  while (lanes < F) lanes *= 2;
  const int64_t nodes = int64_t(1) << depth;
  return nodes * lanes <= kDecidePasses * threads && nodes <= threads &&
         small_staged_use(N, 2 * nodes) + small_decide_use(2 * nodes) <= kScanLds;
}

}  // namespace

// What can be held: a feature's order the registers of one workgroup (8192 rows); the quantiser's workgroup takes
// kQuantChunks chunks; the rows and a slot for each node of a level share the LDS (of 13 levels up to 7732 rows). Up
// to there it is the faster builder of these sizes unless mid_beats_small says otherwise; against the general one:
// 8192 x 20, depth 12 314 us and 806, 8192 x 500, depth 10 483 and 939, 1000 x 10, depth 8 86 and 367.
bool small_tree_fits(int64_t N, int F, int K, int max_depth, int S)
{
  return N <= kSmallMaxRows && K <= kSmallMaxOutputs && N * K <= kQuantChunks * 4096 && max_depth >= 1 &&
         max_depth <= kSmallMaxDepth && small_scan_lds(N, int64_t(1) << (max_depth - 1)) <= kScanLds &&
         S <= LBT_MAX_SPLIT_SAMPLES && static_cast<int64_t>(F) * S < (int64_t(1) << 26) &&
         (static_cast<int64_t>(F) << (max_depth - 1)) <= (int64_t(1) << 22);
}

// All levels in one launch (small_levels_kernel) where a workgroup's look at a level's nodes, which every workgroup has to take for itself, stays
// short: 16,384 lanes for the nodes of the last level, 8192 where a node takes a whole wave. Kernels of a tree and the gaps between them, us, before and
// with one launch: 1000 x 10 depth 8 90 : 61, 500 x 4 depth 3 42 : 32, 4096 x 32 depth 8 135 : 116, 2000 x 32 depth 10 143 : 118,
// 4096 x 64 depth 8 138 : 127; with more lanes 1000 x 64 depth 9 115 : 120, 4096 x 64 depth 10 173 : 199.
bool small_tree_levels_fit(int64_t N, int F, int K, int max_depth)
{
  const int64_t last = int64_t(1) << (max_depth - 1);
  return K == 1 && F <= kSmallDecideFeatures && N <= kDecideRows && max_depth <= kLevelsMaxDepth &&
         (F > 32 ? 64 * last <= 8192 : F > 16 ? 32 * last <= 16384 : 16 * last <= 16384) && small_levels_use(N, max_depth) <= kScanLds;
}

template <typename T>
int small_tree_build(hipStream_t stream, const SmallTreeState& st, const T* X, int64_t row_offset, int64_t N, int F,
                     int K, const double* g, const double* h, const uint8_t* feature_set, const lbt_build_params& prm,
                     double* leaf, int32_t* feature, double* split, double* gain, double* hessian, int32_t* row_leaf,
                     int32_t* n_bins, LevelMeta* level_totals, bool* taken)
{
  *taken = false;
  DeviceAnswer answer;
  LBT_TRY(answer.open(stream));
  PrologueArgs pa;
  pa.row_offset = row_offset;
  pa.N = static_cast<int>(N); pa.F = F; pa.K = K; pa.S = prm.split_samples;
  pa.seed         = prm.seed;
  pa.dataset_rows = prm.dataset_rows;
  pa.g = g; pa.h = h; pa.first_level = prm.abs_sum_chunks;
  pa.l1 = prm.l1_regularization; pa.l2 = prm.l2_regularization;
  pa.max_nodes = prm.max_nodes;
  pa.max_depth = prm.max_depth;
  pa.leaf = leaf; pa.feature = feature; pa.split = split; pa.gain = gain; pa.hessian = hessian;
  pa.answer = answer.words;
  pa.tag    = answer.tag;
  {
    ProfScope ps(LBT_PROF_PROPOSALS, stream);
    static std::atomic<bool> attr_set[kMaxDevices] = {};
    LBT_TRY(allow_dynamic_lds(small_prologue_kernel<T>, 120 * 1024, attr_set));
    int P = 1;
    while (P < prm.split_samples) P <<= 1;
    const size_t feature_lds = static_cast<size_t>(P) * (kProposalScratch<T> + 4) + 16 + N * 4 + 16;
    const size_t quant_lds   = (2048 + 2 * kQuantChunks + 4 + 2 * static_cast<size_t>(K)) * 8;
    const int64_t clear      = std::max<int64_t>(static_cast<int64_t>(prm.max_nodes) * K, N);
    const int64_t words      = st.sync != nullptr ? 3 * static_cast<int64_t>(prm.max_nodes / 2) * F : 0;
    const int clearers       = static_cast<int>(std::min<int64_t>((std::max(clear, words / 4) + kPrologueThreads - 1) / kPrologueThreads, 64));
    small_prologue_kernel<T><<<1 + F + clearers, kPrologueThreads, std::max(feature_lds, quant_lds), stream>>>(X, pa, st);
  }
  if (st.sync != nullptr && level_totals == nullptr) {
    LevelsArgs a;
    a.N = static_cast<int>(N); a.F = F; a.S = prm.split_samples; a.max_depth = prm.max_depth;
    a.lanes_log = kDecideLanes;
    while ((1 << a.lanes_log) < F) a.lanes_log++;
    const size_t lds = small_levels_use(N, prm.max_depth), bins = static_cast<size_t>(F) * st.pitch * sizeof(uint16_t);
    a.all_bins = lds + bins <= kScanLds;
    a.polls    = levels_polls;
    a.leaf = leaf; a.feature = feature; a.split = split; a.gain = gain; a.hessian = hessian; a.row_leaf = row_leaf;
    a.n_bins = answer.words + 1;
    a.tag    = answer.tag;
    a.feature_set = feature_set;
    a.l1 = prm.l1_regularization; a.l2 = prm.l2_regularization; a.min_split_gain = prm.min_split_gain;
    ProfScope ps(LBT_PROF_HISTOGRAM, stream, 0.0, 0);
    const size_t use = lds + (a.all_bins ? bins : 0);
    if (N <= 1024)
      LBT_TRY((launch_small_levels<512, 2>(stream, st, a, use)));
    else if (N <= 2048)
      LBT_TRY((launch_small_levels<1024, 2>(stream, st, a, use)));
    else
      LBT_TRY((launch_small_levels<1024, 4>(stream, st, a, use)));
    LBT_HIP(hipGetLastError());
    unsigned flags = 0;
    LBT_TRY(answer.wait(&flags, n_bins));
    *taken = flags == 0;
    return LBT_OK;
  }
  LevelArgs a;
  a.N = static_cast<int>(N); a.F = F; a.K = K; a.S = prm.split_samples;
  a.feature_set = feature_set;
  a.n_bins = answer.words + 1;
  a.tag    = answer.tag;
  a.l1 = prm.l1_regularization; a.l2 = prm.l2_regularization; a.min_split_gain = prm.min_split_gain;
  a.leaf = leaf; a.feature = feature; a.split = split; a.gain = gain; a.hessian = hessian; a.row_leaf = row_leaf;
  a.lanes_log = kDecideLanes;
  while ((1 << a.lanes_log) < F && a.lanes_log < 6) a.lanes_log++;
  bool decides = false;  // the level's scan has to decide the level above
  int nodes = 0, found = 0;  // the buffers in use
  for (int d = 0; d < prm.max_depth && (d == 0 || !answer.declined()); d++) {
    a.depth       = d;
    a.level_first = static_cast<int>(level_begin(d));
    a.n_nodes     = 1 << d;
    a.last        = d + 1 == prm.max_depth;
    const bool next_decides = next_scan_decides(st, N, F, K, d, prm.max_depth);
    a.node_in    = st.node_of_pos[nodes];
    a.cand_above = st.cand[found];
    a.left_above = st.left[found];
    if (decides) {
      nodes ^= 1;
      found ^= 1;
    }
    a.node_out = st.node_of_pos[nodes];
    a.cand     = st.cand[found];
    a.left     = next_decides ? st.left[found] : nullptr;
    {
      ProfScope ps(LBT_PROF_HISTOGRAM, stream, 0.0, d);
      switch (small_scan_places(N)) {
        case 1024: LBT_TRY((launch_small_scan<256, 4>(stream, st, a, decides))); break;
        case 2048: LBT_TRY((launch_small_scan<512, 4>(stream, st, a, decides))); break;
        case 4096: LBT_TRY((launch_small_scan<1024, 4>(stream, st, a, decides))); break;
        default: LBT_TRY((launch_small_scan<1024, 8>(stream, st, a, decides)));
      }
    }
    decides = next_decides;
    if (level_totals != nullptr) small_count_kernel<<<1, 256, 0, stream>>>(st, a, level_totals + d);
    if (decides) continue;
    ProfScope ps(LBT_PROF_SPLIT, stream);
    // few nodes of many rows near the root, many small ones below
    if ((N >> d) > 1024)
      small_apply_kernel<1024><<<a.n_nodes, 1024, 0, stream>>>(st, a, st.node_of_pos[nodes]);
    else if (d <= 8)
      small_apply_kernel<256><<<a.n_nodes, 256, 0, stream>>>(st, a, st.node_of_pos[nodes]);
    else
      small_apply_kernel<64><<<a.n_nodes, 64, 0, stream>>>(st, a, st.node_of_pos[nodes]);
  }
  LBT_HIP(hipGetLastError());
  unsigned flags = 0;
  LBT_TRY(answer.wait(&flags, n_bins));
  *taken = flags == 0;
  return LBT_OK;
}

template int small_tree_build<float>(hipStream_t, const SmallTreeState&, const float*, int64_t, int64_t, int, int,
                                     const double*, const double*, const uint8_t*, const lbt_build_params&, double*,
                                     int32_t*, double*, double*, double*, int32_t*, int32_t*, LevelMeta*, bool*);
template int small_tree_build<double>(hipStream_t, const SmallTreeState&, const double*, int64_t, int64_t, int, int,
                                      const double*, const double*, const uint8_t*, const lbt_build_params&, double*,
                                      int32_t*, double*, double*, double*, int32_t*, int32_t*, LevelMeta*, bool*);

}  // namespace lbt

void lbt_small_levels_polls(int32_t looks)
{
  lbt::levels_polls = looks < 0 ? lbt::kLevelsPolls : std::min<int>(looks, lbt::kLevelsPolls);  // (a wait is never longer than the library's own)
}
