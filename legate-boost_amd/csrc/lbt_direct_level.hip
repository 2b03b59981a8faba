// Deep levels of a single-output tree without histograms in memory.
//
// With many nodes a level's histograms are far larger than the rows they are made of (1,000,000 x 50 with 512
// samples: 0.84 GB at 2048 nodes against 0.13 GB of records), and clearing, adding, reducing and scanning them took
// 0.74 ms of the 2.7 ms of a depth-12 tree for the last level alone (now 0.24 ms). Here both siblings of every pair are
// accumulated from their rows, but a histogram never leaves the LDS: a workgroup = (node, 16 bytes of a record's
// bins) adds its rows, scans its features' bins and keeps the best split of each. What bounds it is the
// gather of the records and the evaluation of the bins; 64 bins without a row cost one comparison.
//
// Only where every rounded hessian is positive: a scanned histogram is then the running sums everywhere
// (build_tree.cu:645 leaves nothing unscanned) and it does not matter that nothing is derived by subtraction.
#include "lbt_device.h"
#include "lbt_internal.h"

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

template <typename BinT>
__global__ void __launch_bounds__(kDirectThreads) direct_split_kernel(DirectLevel a, int pieces, int width)
{
  constexpr int kPer = 16 / sizeof(BinT);  // features of a workgroup
  extern __shared__ __align__(16) unsigned char smem_raw[];
  unsigned long long* s_hist = reinterpret_cast<unsigned long long*>(smem_raw);  // [kPer][width]
  // the pieces of a node on one XCD, one after the other: they read the same cache lines
  const int j     = static_cast<int>(blockIdx.x >> 3) / pieces * 8 + static_cast<int>(blockIdx.x & 7);
  int piece       = static_cast<int>(blockIdx.x >> 3) % pieces;
  if (j >= a.n_nodes) return;
  const int node   = a.level_first + j;
  const I64Pair ns = a.node_sums[node];
  if (ns.hess <= 0) return;
  int group = 0;
  for (; group < a.n_groups - 1; group++) {
    const int here = (a.rec[group].bins_end + 15) / 16;
    if (piece < here) break;
    piece -= here;
  }
  const RecInfo ri = a.rec[group];
  const int f0 = a.groups[group] + piece * kPer, nf = min(kPer, a.groups[group + 1] - f0);
  const int tid = threadIdx.x, lane = tid & 63;
  for (int i = tid; i < nf * width; i += kDirectThreads) s_hist[i] = 0;
  __syncthreads();
  const unsigned char* const cache = static_cast<const unsigned char*>(a.binned) + ri.base;
  const int begin = a.seg[j], end = a.seg[j + 1];
  for (int i = begin + tid; i < end; i += kDirectThreads) {
    const unsigned char* r = cache + static_cast<int64_t>(a.rows[i]) * ri.stride;
    const uint4 w          = *reinterpret_cast<const uint4*>(r + piece * 16);
    const int2 q           = *reinterpret_cast<const int2*>(r + ri.q_off);
    const unsigned long long word =
      (static_cast<unsigned long long>(static_cast<uint32_t>(q.x)) << 32) | static_cast<uint32_t>(q.y);
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int v = 0; v < kPer; v++)
      if (v < nf) {
        const unsigned bin = sizeof(BinT) == 1 ? (ws[v >> 2] >> (8 * (v & 3))) & 0xffu : (ws[v >> 1 & 3] >> (16 * (v & 1))) & 0xffffu;
        atomicAdd(s_hist + v * width + bin, word);
      }
  }
  __syncthreads();
  const int64_t root = a.node_sums[0].grad, all = (int64_t(1) << 31) + a.n_rows + 1024;
  const int64_t up = (all + root) / 2 + 1, down = (all - root) / 2 + 1;
  const double inv_g = a.scales[2], inv_h = a.scales[3];
  const double reg   = 1e-5 > a.l2 ? 1e-5 : a.l2;
  for (int v = tid >> 6; v < nf; v += kDirectThreads / 64) {
    const int f    = f0 + v;
    const int64_t at = static_cast<int64_t>(j) * a.n_features + f;
    if (a.feature_set != nullptr && a.feature_set[f] == 0) {
      if (lane == 0) a.partial[at] = Cand{0.0, -1};
      continue;
    }
    const int fb = a.row_pointers[f], n_bins = a.row_pointers[f + 1] - fb;
    unsigned long long before = 0, best_left = 0;
    double gain_before = 0.0;  // of the last bin so far: empty bins behind it have the same split
    Cand best{0.0, -1};
    for (int base = 0; base < n_bins; base += 64) {
      const int bin                = base + lane;
      const bool in                = bin < n_bins;
      const unsigned long long add = in ? s_hist[v * width + bin] : 0;
      double gain                  = gain_before;
      unsigned long long left      = before;
      if (__any(add != 0)) {
        left += static_cast<unsigned long long>(wave_inclusive_sum(static_cast<int64_t>(add)));
        const I64Pair ls = unpack_sums(left, up, down);
        bool dead        = false;
        gain             = 0.0;
        add_gain(gain, dead, ls, ns, inv_g, inv_h, a.l1, reg, a.min_split_gain);
        before      = static_cast<unsigned long long>(wave_read_lane(static_cast<int64_t>(left), 63));
        gain_before = __longlong_as_double(wave_read_lane(__double_as_longlong(gain), 63));
      }
      const Cand c{gain, fb + bin};
      if (in && gain > 0 && cand_better(c, best)) {
        best      = c;
        best_left = left;
      }
    }
    for (int off = 32; off >= 1; off >>= 1) {
      const Cand o{__shfl_xor(best.gain, off, 64), __shfl_xor(best.bin, off, 64)};
      const unsigned long long o_left = __shfl_xor(best_left, off, 64);
      if (cand_better(o, best)) {
        best      = o;
        best_left = o_left;
      }
    }
    if (lane == 0) {
      a.partial[at] = best;
      a.left[at]    = unpack_sums(best_left, up, down);
    }
  }
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

int direct_level_launch(hipStream_t stream, const DirectLevel& a, const HistSetup& hs)
{
  const unsigned grid = static_cast<unsigned>((a.n_nodes + 7) / 8 * 8) * static_cast<unsigned>(hs.pieces);
  const size_t lds    = static_cast<size_t>(16 / hs.bin_bytes) * hs.max_bins * sizeof(unsigned long long);
  {
    ProfScope ps(LBT_PROF_HISTOGRAM, stream);
    if (hs.bin_bytes == 1)
      direct_split_kernel<uint8_t><<<grid, kDirectThreads, lds, stream>>>(a, hs.pieces, hs.max_bins);
    else
      direct_split_kernel<uint16_t><<<grid, kDirectThreads, lds, stream>>>(a, hs.pieces, hs.max_bins);
  }
  ProfScope ps(LBT_PROF_SPLIT, stream);
  direct_apply_kernel<<<static_cast<unsigned>((a.n_nodes + 3) / 4), kDirectThreads, 0, stream>>>(a);
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

}  // namespace lbt
