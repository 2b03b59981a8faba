// Deep levels of a single-output tree without histograms in memory.
//
// With many nodes a level's histograms are far larger than the rows they are made of (1,000,000 x 50 with 512
// samples: 0.84 GB at 2048 nodes against 0.13 GB of records), and clearing, adding, reducing and scanning them took
// 0.74 ms of the 2.7 ms of a depth-12 tree for the last level alone (now 0.18 ms). Here both siblings of every pair are
// accumulated from their rows, but a histogram never leaves the LDS: a workgroup = (node, 16 bytes of a record's
// bins) adds its rows, scans its features' bins and keeps the best split of each. What bounds it is the
// gather of the records and the evaluation of the bins; 64 bins without a row cost one comparison.
//
// A tree need not be balanced: with gradients that are mostly noise one node of a level can hold nearly all rows, and
// its few workgroups then were the whole level (1,000,000 x 50 with 512 samples, depth 12, noise: 3.55 ms a tree, where
// histograms in memory took 2.55; 2,000,000 x 80, depth 11 3.93 and 2.14). So the rows of a node of more than two ranges
// of positions are dealt to workgroups by range; each adds its sums to the node's histogram in memory, and the
// last one to finish scans it. It needs 8 bytes per bin and two ranges, in the room of the histograms that are not kept.
// 1,000,000 x 50 with 512 samples, 4 trees of depth 12, us of the launches of levels 9 to 11, with ranges of 8192 and 4096: a
// third of the rows in large nodes 1583 and 1417, nodes of equal size 1193 and 1208, noise 1165 and 1321; 250,000 x 43 with
// 256 samples, noise, 1068 and 889 (2048: half as much again, they add more often).
//
// Only where every rounded hessian is positive: a scanned histogram is then the running sums everywhere
// (build_tree.cu:645 leaves nothing unscanned) and it does not matter that nothing is derived by subtraction.
#include "lbt_device.h"
#include "lbt_internal.h"

#include <type_traits>

namespace lbt {
namespace {

constexpr int kDirectThreads = 256;

// A packed word holds the sum of grads in its upper and of hessians in its lower half. Hessians are not negative and
// sum up to less than 2^32. All |grads| sum up to at most 2^31 + N; with the root's sum G of the grads, sums
// over any rows lie between -(2^31 + N - G) / 2 and (2^31 + N + G) / 2, less than 2^32 apart: a sum that left
// 32 bits is recognised by lying outside.
__device__ __forceinline__ I64Pair unpack_sums(unsigned long long w, int64_t up, int64_t down)
{
  int64_t g = static_cast<int32_t>(static_cast<uint32_t>(w >> 32));
  g += g < -down ? int64_t(1) << 32 : 0;
  g -= g > up ? int64_t(1) << 32 : 0;
  return I64Pair{g, static_cast<int64_t>(static_cast<uint32_t>(w))};
}

// Positions of a range: the shorter ones where their nodes' histograms have the room. A node of up to two ranges is one
// workgroup's, so that a range meets at most two larger ones.
constexpr int kDirectRanges[] = {4096, 8192};

// A thread's next rows: what a piece of their records holds and their pairs. Positions behind the last one read it again.
constexpr int kRowsAtOnce = 4;
struct RowBatch {
  uint4 w[kRowsAtOnce];
  int2 q[kRowsAtOnce];
  __device__ __forceinline__ void load(const DirectLevel& a, const RecInfo& ri, int piece, int i, int end)
  {
    const unsigned char* const cache = static_cast<const unsigned char*>(a.binned) + ri.base;
    int row[kRowsAtOnce];
#pragma unroll
    for (int u = 0; u < kRowsAtOnce; u++) row[u] = a.rows[min(i + u * kDirectThreads, end - 1)];
#pragma unroll
    for (int u = 0; u < kRowsAtOnce; u++) {
      const unsigned char* r = cache + static_cast<int64_t>(row[u]) * ri.stride;
      w[u] = *reinterpret_cast<const uint4*>(r + piece * 16);
      q[u] = *reinterpret_cast<const int2*>(r + ri.q_off);
    }
  }
};

// The rows at positions [begin, end) into the LDS histograms [kPer][width] of the nf features of a
// piece, cleared here. A row is two loads one after the other, its number and its record, and a workgroup of a
// deep level has few rows: four a thread are under way together, the first ones while the histograms are cleared
// (one at a time the levels of 512, 1024 and 2048 nodes of 1,000,000 x 50 took 108, 127 and 193 us, now 92, 108 and 176; two
// at a time the same).
template <typename BinT>
__device__ __forceinline__ void add_rows(const DirectLevel& a, const RecInfo& ri, int piece, int nf, int begin, int end,
                                         int width, unsigned long long* s_hist)
{
  constexpr int kPer  = 16 / sizeof(BinT);
  constexpr int kStep = kRowsAtOnce * kDirectThreads;
  int i = begin + static_cast<int>(threadIdx.x);
  RowBatch batch;
  if (begin < end) batch.load(a, ri, piece, i, end);
  for (int k = threadIdx.x; k < nf * width; k += kDirectThreads) s_hist[k] = 0;
  __syncthreads();
  while (i < end) {
#pragma unroll
    for (int u = 0; u < kRowsAtOnce; u++) {
      if (i + u * kDirectThreads >= end) continue;
      const unsigned long long word =
        (static_cast<unsigned long long>(static_cast<uint32_t>(batch.q[u].x)) << 32) | static_cast<uint32_t>(batch.q[u].y);
      const uint32_t ws[4] = {batch.w[u].x, batch.w[u].y, batch.w[u].z, batch.w[u].w};
#pragma unroll
      for (int v = 0; v < kPer; v++)
        if (v < nf) {
          const unsigned bin = sizeof(BinT) == 1 ? (ws[v >> 2] >> (8 * (v & 3))) & 0xffu : (ws[v >> 1 & 3] >> (16 * (v & 1))) & 0xffffu;
          atomicAdd(s_hist + v * width + bin, word);
        }
    }
    i += kStep;
    if (i < end) batch.load(a, ri, piece, i, end);
  }
  __syncthreads();
}

// Inclusive sums over a wave of packed words. The lower halves' sums stay below 2^32, so nothing is carried and the halves
// are summed on their own, six additions each (64 bits wide hipcc makes five instructions of a step).
__device__ __forceinline__ unsigned long long wave_inclusive_halves(unsigned long long v)
{
  const uint32_t lo = wave_inclusive_sum32(static_cast<uint32_t>(v));
  const uint32_t hi = wave_inclusive_sum32(static_cast<uint32_t>(v >> 32));
  return static_cast<unsigned long long>(hi) << 32 | lo;
}

// A split candidate with what lies left of it, packed. Selects instead of branches: with `if (better) { best = c;
// left = l; }` around the short-circuit comparison hipcc 7.2 kept the old `left` for lanes that had a candidate already.
struct Found {
  double gain;
  int bin;
  unsigned long long left;
  __device__ __forceinline__ void take(double o_gain, int o_bin, unsigned long long o_left, bool valid)
  {
    const int o_rank = o_bin & 511, rank = bin & 511;  // the order of cand_better
    const bool tie    = (o_rank > rank) | ((o_rank == rank) & (o_bin < bin));
    const bool better = valid & (o_bin >= 0) & ((bin < 0) | (o_gain > gain) | ((o_gain == gain) & tie));
    gain = better ? o_gain : gain;
    bin  = better ? o_bin : bin;
    left = better ? o_left : left;
  }
  // the best of a wave's, the same in every lane
  __device__ __forceinline__ Found of_wave() const
  {
    const int from = wave_best_lane(gain, bin);
    if (from < 0) return Found{0.0, -1, 0};
    return Found{wave_read_lane_f64(gain, from), __builtin_amdgcn_readlane(bin, from),
                 static_cast<unsigned long long>(wave_read_lane(static_cast<int64_t>(left), from))};
  }
};

// The best split of one feature, by one wave: every bin's gain as the split evaluation defines it.
__device__ __forceinline__ Found scan_feature(const DirectLevel& a, const I64Pair& ns, int fb, int n_bins, double inv_g,
                                              double inv_h, double reg, int64_t up, int64_t down,
                                              const unsigned long long* s_bins)
{
  const int lane = threadIdx.x & 63;
  unsigned long long before = 0;
  double gain_before = 0.0;  // of the last bin so far: empty bins behind it have the same split
  Found best{0.0, -1, 0};
  for (int base = 0; base < n_bins; base += 64) {
    const int bin                = base + lane;
    const bool in                = bin < n_bins;
    const unsigned long long add = in ? s_bins[bin] : 0;
    double gain                  = gain_before;
    unsigned long long left      = before;
    if (__any(add != 0)) {
      left += wave_inclusive_halves(add);
      const I64Pair ls = unpack_sums(left, up, down);
      bool dead        = false;
      gain             = 0.0;
      add_gain(gain, dead, ls, ns, inv_g, inv_h, a.l1, reg, a.min_split_gain);
      before      = static_cast<unsigned long long>(wave_read_lane(static_cast<int64_t>(left), 63));
      gain_before = wave_read_lane_f64(gain, 63);
    }
    best.take(gain, fb + bin, left, in & (gain > 0));
  }
  return best.of_wave();
}

// Most bins cannot be the best split, and a shorter sum shows it. With integers gl, hl, gr, hr left and right of a bin,
// gl^2 / (hl + reg / inv_h) + gr^2 / (hr + reg / inv_h) times inv_g^2 / inv_h is what the gain is made of without a
// penalty (l1 = 0). Formed in 32 bits, every term but the sums rounded once (2^-24) and one approximate reciprocal (2^-23), it
// is right to 15 * 2^-24 < 2^-20: nothing is subtracted after the exact whole-number differences.
// The gain is a monotone function of the two quotients' sum, and every rounding on the way to it (minus the node's own
// term, minus a min_split_gain that is not negative, where it ends above 0) merges sums within a few units of 2^-52: so a
// bin whose estimate is below 1 - 2^-18 of the feature's largest has a smaller gain. One gain per lane is then
// formed exactly, of its largest estimate, and where a lane holds a second one that near (equal columns) the feature
// is scanned as above. A bin without rows has the sums of the last one with rows before it: only those are
// estimated, and which of the bins up to the next one with rows the tie rule takes is worked out for the best.
// A lane takes four bins in a row, so that a running sum over the lanes serves 256 bins; one where they are at most 64, of which
// four a lane would leave three lanes of four idle (the four levels of 60,000 x 200 with 64 samples, depth 11: 275 us with four, and
// a tree 949; 909 with one).
// The 12 launches of levels 9 to 11 of four trees of depth 12, 1,000,000 x 50 with 512 samples: 1361 us with estimates in
// 64 bits of one bin a lane, now 1208; what bounds them then is the chain of loads of a workgroup's rows (75 of the 82 us of
// level 9 without any scan).
// Not used with magnitudes whose products might leave the range of 32-bit floats: whole numbers are below 2^33, extra
// (reg / inv_h) below 2^40.
constexpr float kNearBest = 1.0f - 1.0f / (1 << 18);
__device__ __forceinline__ bool estimates_hold(const DirectLevel& a, double inv_g, double inv_h, double reg)
{
  auto ordinary = [](double v) { return v >= 1e-60 && v <= 1e60; };
  return a.l1 == 0.0 && a.min_split_gain >= 0.0 && ordinary(inv_g) && ordinary(inv_h) && ordinary(reg) &&
         reg / inv_h >= 1e-30 && reg / inv_h <= 1e12;
}

// kSmall: all sums of grads fit 32 bits with their sign. kBins: bins in a row of a lane
template <bool kSmall, int kBins>
__device__ __forceinline__ Found scan_feature_estimated(const DirectLevel& a, const I64Pair& ns, int fb, int n_bins,
                                                        double inv_g, double inv_h, double reg, int64_t up,
                                                        int64_t down, const unsigned long long* s_bins)
{
  static_assert(kBins == 1 || kBins == 4);
  const int lane        = threadIdx.x & 63;
  const float extra     = static_cast<float>(reg / inv_h);
  const int small_g     = static_cast<int>(ns.grad);
  const double all_g    = static_cast<double>(ns.grad);
  const uint32_t all_h  = static_cast<uint32_t>(ns.hess);
  // grads lie in [-down, up] and up + down < 2^32: the lower 32 bits of grad + down are grad + down
  const uint32_t down32  = static_cast<uint32_t>(down);
  const double down_sums = static_cast<double>(down);
  uint32_t before_g = 0, before_h = 0, left_g = 0, left_h = 0;
  float most = -1.0f, second = -1.0f;  // of this lane the two largest estimates
  int bin_1  = 0;
  for (int base = 0; base < n_bins; base += 64 * kBins) {
    const int first = base + lane * kBins;
    uint32_t g[kBins] = {}, h[kBins] = {};
    if (kBins == 1 && first < n_bins) {
      const unsigned long long w = s_bins[first];
      h[0] = static_cast<uint32_t>(w), g[0] = static_cast<uint32_t>(w >> 32);
    } else if (kBins == 4 && first < n_bins) {
      // (a feature's bins take a multiple of four places, zeros behind the last one)
      const uint4 w0 = *reinterpret_cast<const uint4*>(s_bins + first), w1 = *reinterpret_cast<const uint4*>(s_bins + first + 2);
      h[0] = w0.x, g[0] = w0.y, h[1 % kBins] = w0.z, g[1 % kBins] = w0.w;
      h[2 % kBins] = w1.x, g[2 % kBins] = w1.y, h[3 % kBins] = w1.z, g[3 % kBins] = w1.w;
    }
    // The lower halves' sums stay below 2^32, so nothing is carried and the halves are summed on their own.
    uint32_t sum_g = 0, sum_h = 0;
#pragma unroll
    for (int u = 0; u < kBins; u++) sum_g += g[u], sum_h += h[u];
    if (!__any(sum_h != 0)) continue;
    const uint32_t to_g = before_g + wave_inclusive_sum32(sum_g);
    const uint32_t to_h = before_h + wave_inclusive_sum32(sum_h);
    before_g = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(to_g), 63));
    before_h = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(to_h), 63));
    uint32_t lg = to_g - sum_g, lh = to_h - sum_h;
#pragma unroll
    for (int u = 0; u < kBins; u++) {
      lg += g[u];
      lh += h[u];
      float gl, gr;
      if constexpr (kSmall) {
        gl = static_cast<float>(static_cast<int>(lg));
        gr = static_cast<float>(small_g - static_cast<int>(lg));
      } else {
        const double left = static_cast<double>(lg + down32) - down_sums;
        gl = static_cast<float>(left);
        gr = static_cast<float>(all_g - left);
      }
      const float pl = static_cast<float>(lh) + extra, pr = static_cast<float>(all_h - lh) + extra;
      const float sum      = __builtin_fmaf(gl * gl, pr, gr * gr * pl) * __builtin_amdgcn_rcpf(pl * pr);
      const float estimate = ((h[u] != 0) & (lh != all_h)) ? sum : -1.0f;
      const bool more      = estimate > most;
      second = __builtin_fmaxf(second, __builtin_fminf(most, estimate));
      most   = __builtin_fmaxf(most, estimate);
      left_g = more ? lg : left_g;
      left_h = more ? lh : left_h;
      bin_1  = more ? first + u : bin_1;
    }
  }
  // positive floats compare as whole numbers; an estimate of 0 is a gain that is not positive
  const uint32_t top = wave_max_u32(most > 0.0f ? __float_as_uint(most) : 0u);
  if (top == 0) return Found{0.0, -1, 0};  // no valid split
  const float near = __uint_as_float(top) * kNearBest;
  if (__any(second >= near)) return scan_feature(a, ns, fb, n_bins, inv_g, inv_h, reg, up, down, s_bins);
  const unsigned long long left = static_cast<unsigned long long>(left_g) << 32 | left_h;
  bool dead   = false;
  double gain = 0.0;
  add_gain(gain, dead, unpack_sums(left, up, down), ns, inv_g, inv_h, a.l1, reg, a.min_split_gain);
  const bool maybe = most >= near && gain > 0;
  int pick = -1;
  for (unsigned long long left_to_do = __ballot(maybe); left_to_do != 0; left_to_do &= left_to_do - 1) {
    const int from = __builtin_ctzll(left_to_do), bin = __builtin_amdgcn_readlane(bin_1, from);
    int next = n_bins;  // the next bin with rows
    for (int base = bin + 1; base < n_bins; base += 64) {
      const unsigned long long rows = __ballot(base + lane < n_bins && static_cast<uint32_t>(s_bins[min(base + lane, n_bins - 1)]) != 0);
      if (rows != 0) {
        next = base + __builtin_ctzll(rows);
        break;
      }
    }
    // of bins that share a gain the one of 511 mod 512, else the last one
    if (lane == from) pick = min((fb + bin) | 511, fb + next - 1);
  }
  return Found{gain, pick, left}.of_wave();
}

// The best split of each of the features [f0, f0 + nf) of node j from its histograms in the LDS.
__device__ __forceinline__ void scan_features(const DirectLevel& a, int j, const I64Pair& ns, int f0, int nf, int width,
                                              const unsigned long long* s_hist)
{
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int64_t root = a.node_sums[0].grad, all = (int64_t(1) << 31) + a.n_rows + 1024;
  const int64_t up = (all + root) / 2 + 1, down = (all - root) / 2 + 1;
  const double inv_g = a.scales[2], inv_h = a.scales[3];
  const double reg   = 1e-5 > a.l2 ? 1e-5 : a.l2;
  const bool estimated = estimates_hold(a, inv_g, inv_h, reg);
  const bool small     = up <= 2147483647LL && down <= 2147483647LL;
  for (int v = wave; v < nf; v += kDirectThreads / 64) {
    const int f    = f0 + v;
    const int64_t at = static_cast<int64_t>(j) * a.n_features + f;
    if (a.feature_set != nullptr && a.feature_set[f] == 0) {
      if (lane == 0) a.partial[at] = Cand{0.0, -1};
      continue;
    }
    const int fb = a.row_pointers[f], n_bins = a.row_pointers[f + 1] - fb;
    const unsigned long long* bins = s_hist + v * width;
    auto estimate    = [&](auto small_c) {
      constexpr bool kSmall = decltype(small_c)::value;
      return n_bins <= 64 ? scan_feature_estimated<kSmall, 1>(a, ns, fb, n_bins, inv_g, inv_h, reg, up, down, bins)
                          : scan_feature_estimated<kSmall, 4>(a, ns, fb, n_bins, inv_g, inv_h, reg, up, down, bins);
    };
    const Found best = !estimated ? scan_feature(a, ns, fb, n_bins, inv_g, inv_h, reg, up, down, bins)
                       : small    ? estimate(std::true_type{})
                                  : estimate(std::false_type{});
    if (lane == 0) {
      a.partial[at] = Cand{best.gain, best.bin};
      a.left[at]    = unpack_sums(best.left, up, down);
    }
  }
}

// Piece `part` of all records' pieces: its record group, its number there, its first feature and how many.
struct Piece {
  RecInfo rec;
  int number, f0, nf;
};
template <typename BinT>
__device__ __forceinline__ Piece piece_of(const DirectLevel& a, int part)
{
  constexpr int kPer = 16 / sizeof(BinT);
  int group          = 0;
  for (; group < a.n_groups - 1; group++) {
    const int here = (a.rec[group].bins_end + 15) / 16;
    if (part < here) break;
    part -= here;
  }
  const int f0 = a.groups[group] + part * kPer;
  return Piece{a.rec[group], part, f0, min(kPer, a.groups[group + 1] - f0)};
}

// The large nodes that lie in a range of positions: one may hold its first position, one may begin inside and go on
// behind it. What the range adds of a node goes to the node's histogram in memory; the last of its ranges to arrive
// finds the splits.
template <typename BinT>
__device__ __forceinline__ void add_range(const DirectLevel& a, int range, int part, int pieces, int width,
                                          unsigned long long* s_hist)
{
  constexpr int kPer = 16 / sizeof(BinT);
  const int tid   = threadIdx.x;
  const int first = range * a.range;
  const int last  = static_cast<int>(min(a.n_rows, static_cast<int64_t>(first) + a.range));
  for (int side = 0; side < 2; side++) {
    const int j = side == 0 ? a.block_seg[first / a.slab] : (last < a.n_rows ? a.block_seg[last / a.slab] : -1);
    if (j < 0) continue;
    const int begin = a.seg[j], end = a.seg[j + 1];
    if (end - begin <= 2 * a.range || (side == 1 && (begin <= first || begin >= last))) continue;
    const Piece p = piece_of<BinT>(a, part);
    add_rows<BinT>(a, p.rec, p.number, p.nf, max(first, begin), min(last, end), width, s_hist);
    // large nodes begin more than two ranges apart: a slot each. Slots and counters are zero between nodes.
    const int64_t slot      = static_cast<int64_t>(begin / (2 * a.range)) * pieces + part;
    unsigned long long* sum = a.large + slot * kPer * width;
    for (int i = tid; i < p.nf * width; i += kDirectThreads)
      if (s_hist[i] != 0) atomicAdd(sum + i, s_hist[i]);
    // What orders these adds before the last arriver's loads is the target, not the memory model of the language, in which all of them are
    // relaxed: (1) vmcnt counts an atomic without result until it has been performed at the scope it was asked with, so behind the wait
    // and the barrier all waves' adds are where the whole device sees them before the workgroup is counted; (2) a load at
    // device scope is not answered from a cache of its own XCD that could be stale. The slot is cleared by plain stores: nothing
    // touches it again within the launch, and its end writes them back.
    // The model's own means, us of the launches of levels 9 to 11 of 1,000,000 x 50 with 512 samples, noise, and of 2,000,000 x 80,
    // depth 11: as here 341 and 184; one thread's release (it writes the whole L2 back) and the last arriver's acquire 516 and
    // 313; the acquire alone, which orders nothing without the release, 356 and 187.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "written for what gfx950 guarantees of waited atomics and of loads at device scope"
#endif
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // (the answer goes through the histograms' LDS: a word more and only four workgroups of 512 bins share a CU)
    if (tid == 0) {
      const int ranges = (end - 1) / a.range - begin / a.range + 1;
      s_hist[0]        = atomicAdd(a.arrivals + slot, 1) + 1 == ranges ? 1 : 0;
    }
    __syncthreads();
    const bool last_of_node = s_hist[0] != 0;
    __syncthreads();
    if (!last_of_node) continue;
    for (int i = tid; i < p.nf * width; i += kDirectThreads) {
      s_hist[i] = __hip_atomic_load(sum + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      sum[i]    = 0;
    }
    if (tid == 0) a.arrivals[slot] = 0;
    __syncthreads();
    scan_features(a, j, a.node_sums[a.level_first + j], p.f0, p.nf, width, s_hist);
    __syncthreads();
  }
}

// Workgroups [0, large_blocks): (range of positions, piece), the parts of large nodes that lie in it. The others:
// (node, piece), the smaller nodes. The pieces of a range (a node) on one XCD, one after the other: they read the same
// cache lines.
template <typename BinT>
__global__ void __launch_bounds__(kDirectThreads)
  direct_split_kernel(DirectLevel a, int pieces, int width, int ranges, int large_blocks)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  unsigned long long* s_hist = reinterpret_cast<unsigned long long*>(smem_raw);  // [16 / sizeof(BinT)][width]
  if (static_cast<int>(blockIdx.x) < large_blocks) {
    const int id = static_cast<int>(blockIdx.x), range = (id >> 3) / pieces * 8 + (id & 7);
    if (range < ranges) add_range<BinT>(a, range, (id >> 3) % pieces, pieces, width, s_hist);
    return;
  }
  const int id = static_cast<int>(blockIdx.x) - large_blocks;
  const int j  = (id >> 3) / pieces * 8 + (id & 7);
  if (j >= a.n_nodes) return;
  const I64Pair ns = a.node_sums[a.level_first + j];
  const int begin = a.seg[j], end = a.seg[j + 1];
  if (ns.hess <= 0 || end - begin > 2 * a.range) return;
  const Piece p = piece_of<BinT>(a, (id >> 3) % pieces);
  add_rows<BinT>(a, p.rec, p.number, p.nf, begin, end, width, s_hist);
  scan_features(a, j, ns, p.f0, p.nf, width, s_hist);
}

// The best feature of every node and what follows from it (build_tree.cu:740-782), one wave per node.
__global__ void __launch_bounds__(kDirectThreads) direct_apply_kernel(DirectLevel a)
{
  const int j = static_cast<int>((blockIdx.x * kDirectThreads + threadIdx.x) >> 6), lane = threadIdx.x & 63;
  if (j >= a.n_nodes) return;
  const int node   = a.level_first + j;
  const I64Pair ns = a.node_sums[node];
  if (ns.hess <= 0) return;
  Cand best{0.0, -1};
  int ft = 0;
  for (int f = lane; f < a.n_features; f += 64) {
    const Cand o = a.partial[static_cast<int64_t>(j) * a.n_features + f];
    if (cand_better(o, best)) {
      best = o;
      ft   = f;
    }
  }
  for (int off = 32; off >= 1; off >>= 1) {
    const Cand o{__shfl_xor(best.gain, off, 64), __shfl_xor(best.bin, off, 64)};
    const int of = __shfl_xor(ft, off, 64);
    if (cand_better(o, best)) {
      best = o;
      ft   = of;
    }
  }
  if (lane != 0 || !(best.bin >= 0 && best.gain > 1e-5)) return;
  const double inv_g = a.scales[2], inv_h = a.scales[3];
  const I64Pair ls = a.left[static_cast<int64_t>(j) * a.n_features + ft];
  const I64Pair rs{ns.grad - ls.grad, ns.hess - ls.hess};
  const int lc = left_child(node), rc = right_child(node);
  a.node_sums[lc]   = ls;
  a.node_sums[rc]   = rs;
  a.leaf[lc]        = calculate_leaf_value(static_cast<double>(ls.grad) * inv_g, static_cast<double>(ls.hess) * inv_h, a.l1, a.l2);
  a.leaf[rc]        = calculate_leaf_value(static_cast<double>(rs.grad) * inv_g, static_cast<double>(rs.hess) * inv_h, a.l1, a.l2);
  a.feature[node]   = ft;
  a.split[node]     = a.proposals[best.bin];
  a.gain[node]      = best.gain;
  a.split_bin[node] = best.bin - a.row_pointers[ft];
}

}  // namespace

// Words of a feature's histogram: the scan takes four bins a lane
static int direct_width(const HistSetup& hs) { return (hs.max_bins + 3) / 4 * 4; }

static size_t direct_large_words(const HistSetup& hs, int64_t n_rows, int range)
{
  return n_rows <= 2 * range ? 0 : static_cast<size_t>(n_rows / (2 * range) + 1) * hs.pieces * (16 / hs.bin_bytes) * direct_width(hs);
}

size_t direct_large_bytes(const HistSetup& hs, int64_t n_rows, int range)
{
  const size_t counters = static_cast<size_t>(n_rows / (2 * range) + 1) * hs.pieces * sizeof(int32_t);
  return n_rows <= 2 * range ? 0 : direct_large_words(hs, n_rows, range) * sizeof(unsigned long long) + (counters + 15) / 16 * 16;
}

int direct_range(const HistSetup& hs, int64_t n_rows, size_t room)
{
  for (const int range : kDirectRanges)
    if (direct_large_bytes(hs, n_rows, range) <= room) return range;
  return 0;
}

int direct_level_launch(hipStream_t stream, DirectLevel a, const HistSetup& hs)
{
  LBT_REQUIRE(a.range > 0 && a.range % a.slab == 0, "ranges of positions are whole slabs");
  a.arrivals          = reinterpret_cast<int32_t*>(a.large + direct_large_words(hs, a.n_rows, a.range));
  const int ranges    = a.n_rows <= 2 * a.range ? 0 : ceil_div(a.n_rows, a.range);
  const int large     = (ranges + 7) / 8 * 8 * hs.pieces;
  const int width     = direct_width(hs);
  const unsigned grid = static_cast<unsigned>(large) + static_cast<unsigned>((a.n_nodes + 7) / 8 * 8) * static_cast<unsigned>(hs.pieces);
  const size_t lds    = static_cast<size_t>(16 / hs.bin_bytes) * width * sizeof(unsigned long long);
  {
    ProfScope ps(LBT_PROF_HISTOGRAM, stream);
    if (hs.bin_bytes == 1)
      direct_split_kernel<uint8_t><<<grid, kDirectThreads, lds, stream>>>(a, hs.pieces, width, ranges, large);
    else
      direct_split_kernel<uint16_t><<<grid, kDirectThreads, lds, stream>>>(a, hs.pieces, width, ranges, large);
  }
  ProfScope ps(LBT_PROF_SPLIT, stream);
  direct_apply_kernel<<<static_cast<unsigned>((a.n_nodes + 3) / 4), kDirectThreads, 0, stream>>>(a);
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

}  // namespace lbt
