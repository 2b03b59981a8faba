// The steps of a boosting round either side of the tree build: the weighted gradient
// (legateboost/legateboost.py:189-224 with objectives.py:131-147 and :489-531), the
// prediction update from the rows' leaves (legateboost.py:268), and the row gather of
// src/utils/gather.cu:26-91. All of it is streaming work over [n_rows][n_outputs] doubles:
// one read of every input, one write of every output.
#include <algorithm>
#include <iterator>
#include <limits>
#include <type_traits>

#include "lbt_internal.h"

namespace lbt {

constexpr int kMaskFeatures = 8192;  // bits of a launch's arguments
constexpr int kBoostThreads = 256;
// A tree's leaf values, to be added to the predictions (add_leaf_values_kernel) where their gradients are formed. Bound by memory for
// many rows: the predictions are not read again (10,000,000 rows with the chunk sums: 42 and 59 us, now 73; 94 with one entry's loads
// behind the store of the one before). For few a launch less a round: a fit of 12 rounds of 1000 x 10 f64 900 us, now 880.
struct LeafAdd {
  const double* leaf;  // null: the predictions stay as they are
  int n_nodes;
  const int32_t* row_leaf;
};
template <bool kAdds>
__device__ __forceinline__ double prediction_at(const LeafAdd& a, const double* pred, int64_t i, int K)
{
  const double p = pred[i];
  if constexpr (!kAdds) return p;
  const int64_t r  = K == 1 ? i : i / K;
  const int node   = a.row_leaf[r];
  const bool known = node >= 0 && node < a.n_nodes;  // a row of no leaf keeps its prediction, whatever its bits
  const double v   = a.leaf[static_cast<int64_t>(known ? node : 0) * K + (i - r * K)];
  return known ? p + v : p;
}

// One element per thread: squared error (any number of outputs) and log loss with one output.
template <bool kLogistic, bool kAdds>
__global__ void __launch_bounds__(kBoostThreads)
  gradient_elementwise_kernel(LeafAdd add, double* __restrict__ pred, const double* __restrict__ y,
                              const double* __restrict__ weight, double lr, int64_t n, int K,
                              double* __restrict__ g, double* __restrict__ h)
{
  const int64_t i = blockIdx.x * static_cast<int64_t>(kBoostThreads) + threadIdx.x;
  if (i >= n) return;
  const double w = weight != nullptr ? weight[K == 1 ? i : i / K] : 1.0;
  double p = prediction_at<kAdds>(add, pred, i, K), h0 = 1.0;
  if (kAdds) pred[i] = p;
  if (kLogistic) {
    p  = 1.0 / (1.0 + exp(-p));
    h0 = p * (1.0 - p);
  }
  double go, ho;
  weigh(p - y[i], h0, w, lr, &go, &ho);
  g[i] = go;
  h[i] = ho;
}

// One row per thread: softmax over the row's K outputs, then the class gradient.
// kCols > 0 keeps the row in registers; 0 recomputes the exponentials instead. See softmax_by_entry.
template <int kCols>
__global__ void __launch_bounds__(kBoostThreads)
  gradient_softmax_rows_kernel(const double* __restrict__ pred, const double* __restrict__ y,
                               const double* __restrict__ weight, double lr, int64_t n_rows, int K,
                               double* __restrict__ g, double* __restrict__ h)
{
  const int64_t r = blockIdx.x * static_cast<int64_t>(kBoostThreads) + threadIdx.x;
  if (r >= n_rows) return;
  const double w  = weight != nullptr ? weight[r] : 1.0;
  const int label = static_cast<int>(y[r]);
  const double* p = pred + r * K;
  double* go      = g + r * K;
  double* ho      = h + r * K;
  if (kCols > 0) {
    double e[kCols > 0 ? kCols : 1];
    double top = p[0];
#pragma unroll
    for (int k = 0; k < kCols; k++) {
      e[k] = p[k];
      top  = fmax(top, e[k]);
    }
    double div = 0.0;
#pragma unroll
    for (int k = 0; k < kCols; k++) {
      e[k] = exp(e[k] - top);
      div += e[k];
    }
#pragma unroll
    for (int k = 0; k < kCols; k++) {
      const double q = e[k] / div;
      weigh(k == label ? q + -1.0 : q, q * (1.0 - q), w, lr, go + k, ho + k);
    }
  } else {
    double top = p[0];
    for (int k = 1; k < K; k++) top = fmax(top, p[k]);
    double div = 0.0;
    for (int k = 0; k < K; k++) div += exp(p[k] - top);
    for (int k = 0; k < K; k++) {
      const double q = exp(p[k] - top) / div;
      weigh(k == label ? q + -1.0 : q, q * (1.0 - q), w, lr, go + k, ho + k);
    }
  }
}

// The same gradients together with the first level of the quantiser's two absolute sums
// (build_tree.cu:77-83 sums |g| and |h| over all entries before it rounds any of them): the
// gradient pass already holds every entry in registers, so the sums cost no second read of g
// and h. The order of the sums is the quantiser's fixed one: chunk c covers the 4096 flat
// entries [4096 c, 4096 c + 4096), lane t adds entries t, t + 256, ... in ascending order, a
// binary tree (strides 128 .. 1) joins the 256 lanes. One workgroup per chunk.
constexpr int kSumChunk = 4096;
static_assert(kSumChunk == 16 * kBoostThreads, "a lane adds 16 entries of a chunk");

__device__ inline void store_chunk_sums(double xa, double xb, double* sa, double* sb, double* out_a, double* out_b)
{
  sa[threadIdx.x] = xa;
  sb[threadIdx.x] = xb;
  __syncthreads();
  for (int stride = kBoostThreads / 2; stride >= 1; stride >>= 1) {
    if (static_cast<int>(threadIdx.x) < stride) {
      sa[threadIdx.x] += sa[threadIdx.x + stride];
      sb[threadIdx.x] += sb[threadIdx.x + stride];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out_a[blockIdx.x] = sa[0];
    out_b[blockIdx.x] = sb[0];
  }
}

template <bool kLogistic, bool kAdds>
__global__ void __launch_bounds__(kBoostThreads)
  gradient_elementwise_sums_kernel(LeafAdd add, double* __restrict__ pred, const double* __restrict__ y,
                                   const double* __restrict__ weight, double lr, int64_t n, int K,
                                   double* __restrict__ g, double* __restrict__ h, double* __restrict__ sum_g,
                                   double* __restrict__ sum_h)
{
  __shared__ double sa[kBoostThreads];
  __shared__ double sb[kBoostThreads];
  double xa = 0.0, xb = 0.0;
  // four entries' values are asked for before the first of them is stored
  constexpr int kTogether = 4;
  for (int j0 = 0; j0 < kSumChunk / kBoostThreads; j0 += kTogether) {
    const int64_t first = blockIdx.x * static_cast<int64_t>(kSumChunk) + threadIdx.x + static_cast<int64_t>(kBoostThreads) * j0;
    double p[kTogether], target[kTogether], w[kTogether];
#pragma unroll
    for (int u = 0; u < kTogether; u++) {
      const int64_t i = min(first + kBoostThreads * u, n - 1);
      p[u]      = prediction_at<kAdds>(add, pred, i, K);
      target[u] = y[i];
      w[u]      = weight != nullptr ? weight[K == 1 ? i : i / K] : 1.0;
    }
#pragma unroll
    for (int u = 0; u < kTogether; u++) {
      const int64_t i = first + kBoostThreads * u;
      if (i >= n) continue;
      if (kAdds) pred[i] = p[u];
      double q = p[u], h0 = 1.0;
      if (kLogistic) {
        q  = 1.0 / (1.0 + exp(-q));
        h0 = q * (1.0 - q);
      }
      double go, ho;
      weigh(q - target[u], h0, w[u], lr, &go, &ho);
      g[i] = go;
      h[i] = ho;
      xa += fabs(go);
      xb += fabs(ho);
    }
  }
  store_chunk_sums(xa, xb, sa, sb, sum_g, sum_h);
}

// Softmax of rows of up to kSoftmaxCols outputs: a thread has entries, and only the row's maximum and the sum of its exponentials are a
// row's work, which a thread each does from the LDS, in the order of the outputs. Bound by memory: pred is read and g and h are written in whole
// lines (a thread with a row of 8 outputs met 64 lines with each load and store), and with kSums the pass that sums |g| and |h| is
// none of its own. A stage is kSumStage entries: with kSums lane t's entries t + 256 j of a chunk's first stage are its j = 0 .. 7, those of the
// second its j = 8 .. 15; without it a workgroup has one stage. Rows that straddle two stages have their other outputs read, and their
// exponentials formed, for each of them.
constexpr int kSumStage    = 2048;
constexpr int kSoftmaxCols = 128;
constexpr int kStageTurns  = kSumStage / kBoostThreads;
// a place behind every row of a multiple of four outputs: a thread with a row meets other banks than its neighbours
constexpr int kStagePlaces = kSumStage * 5 / 4 + 3 * kSoftmaxCols;
constexpr int kStageRows   = kSumStage / 2 + 2;
static_assert(2 * kSoftmaxCols <= kBoostThreads, "the outputs of straddling rows are one a thread");
template <bool kSums>
__global__ void __launch_bounds__(kBoostThreads)
  gradient_softmax_kernel(const double* __restrict__ pred, const double* __restrict__ y, const double* __restrict__ weight, double lr,
                          int64_t n_rows, int K, double* __restrict__ g, double* __restrict__ h, double* __restrict__ sum_g,
                          double* __restrict__ sum_h)
{
  __shared__ double s_p[kStagePlaces];
  __shared__ double s_row[kStageRows];
  static_assert(kStagePlaces >= 2 * kBoostThreads, "the chunk's sums are formed in the same place");
  const int tid       = static_cast<int>(threadIdx.x);
  const int64_t n     = n_rows * K;
  const unsigned inverse = ((1u << 20) + static_cast<unsigned>(K) - 1) / static_cast<unsigned>(K);  // i / K for i below a stage and two rows
  const int pad       = K % 4 == 0 ? 1 : 0;
  double xa = 0.0, xb = 0.0;
  for (int stage = 0; stage < (kSums ? kSumChunk / kSumStage : 1); stage++) {
    const int64_t e0 = (blockIdx.x * static_cast<int64_t>(kSums ? kSumChunk / kSumStage : 1) + stage) * kSumStage;
    if (e0 >= n) break;
    const int64_t r0 = e0 / K, f0 = r0 * K;
    const int front = static_cast<int>(e0 - f0);                                   // outputs of the first row that lie before the stage
    const int in    = static_cast<int>(n - e0 < kSumStage ? n - e0 : kSumStage);   // entries of the stage
    const int rows  = static_cast<int>(static_cast<unsigned>(front + in + K - 1) * inverse >> 20);
    const int back  = rows * K - front - in;                                       // of the last row behind it
    double p[kStageTurns], w[kStageTurns];
    int at[kStageTurns], row[kStageTurns];  // place in the LDS, row of the stage
    unsigned hits = 0;                      // bit j: the entry is that of its row's label
#pragma unroll
    for (int j = 0; j < kStageTurns; j++) {
      const int i = front + min(tid + kBoostThreads * j, in - 1);
      p[j]        = pred[f0 + i];
      row[j]      = static_cast<int>(static_cast<unsigned>(i) * inverse >> 20);
      hits |= (static_cast<int>(y[r0 + row[j]]) == i - row[j] * K ? 1u : 0u) << j;
      w[j]        = weight != nullptr ? weight[r0 + row[j]] : 1.0;
      at[j]       = i + row[j] * pad;
    }
    const bool extra = tid < front + back;
    const int xi     = extra ? (tid < front ? tid : tid + in) : 0;
    const int xrow   = static_cast<int>(static_cast<unsigned>(xi) * inverse >> 20);
    double xp        = pred[f0 + xi];
    if (stage > 0) __syncthreads();  // the rows' sums before are still read
#pragma unroll
    for (int j = 0; j < kStageTurns; j++)
      if (tid + kBoostThreads * j < in) s_p[at[j]] = p[j];
    if (extra) s_p[xi + xrow * pad] = xp;
    __syncthreads();
    for (int r = tid; r < rows; r += kBoostThreads) {
      const double* const of = s_p + r * (K + pad);
      double top = of[0];
      for (int k = 1; k < K; k++) top = fmax(top, of[k]);
      s_row[r] = top;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kStageTurns; j++) {
      p[j] = exp(p[j] - s_row[row[j]]);
      if (tid + kBoostThreads * j < in) s_p[at[j]] = p[j];
    }
    if (extra) s_p[xi + xrow * pad] = exp(xp - s_row[xrow]);
    __syncthreads();
    for (int r = tid; r < rows; r += kBoostThreads) {
      const double* const of = s_p + r * (K + pad);
      double div = 0.0;
      for (int k = 0; k < K; k++) div += of[k];
      s_row[r] = div;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kStageTurns; j++) {
      const int i = tid + kBoostThreads * j;
      if (i < in) {
        const double q = p[j] / s_row[row[j]];
        double go, ho;
        weigh((hits >> j & 1) != 0 ? q + -1.0 : q, q * (1.0 - q), w[j], lr, &go, &ho);
        g[e0 + i] = go;
        h[e0 + i] = ho;
        xa += fabs(go);
        xb += fabs(ho);
      }
    }
  }
  if constexpr (kSums) {
    __syncthreads();
    store_chunk_sums(xa, xb, s_p, s_p + kBoostThreads, sum_g, sum_h);
  }
}

// us with a thread for an entry and one for a row: 16,000,000 entries in rows of 2 83 : 78, of 4 78 : 80, of 8 75 : 103, of 16 74 : 129;
// 5,000,000 of 5 24.8 : 26.1, of 8 23 : 31; 1,280,000 of 5 10.6 : 8.9, of 8 10.0 : 10.6; 20,000 of 8 5.3 : 3.1. Rows that are not held in registers
// never: 20,000 of 9 5.4 : 7.4, 16,000,000 75 : 598, of 20 75 : 1108, of 64 77 : 802.
inline bool softmax_by_entry(int64_t n, int K)
{
  const bool in_registers = K <= 8 || K == 10 || K == 16;
  return K <= kSoftmaxCols && (!in_registers || (K >= 5 && n >= 4000000));
}

// The same for rows of more outputs: a workgroup computes the rows that meet its chunk of entries (a row that straddles
// two stages or chunks is computed for each of them, which stores the same values), keeps the
// entries in the LDS and adds them up from there in the quantiser's order. The chunk is taken
// in stages of 2048 entries: lane t's entries t + 256 j of the first stage are its j = 0 .. 7,
// those of the second its j = 8 .. 15, so the order of its sum is the same.
__global__ void __launch_bounds__(kBoostThreads)
  gradient_softmax_rows_sums_kernel(const double* __restrict__ pred, const double* __restrict__ y,
                                    const double* __restrict__ weight, double lr, int64_t n_rows, int K,
                                    double* __restrict__ g, double* __restrict__ h, double* __restrict__ sum_g,
                                    double* __restrict__ sum_h)
{
  __shared__ double s_g[kSumStage];
  __shared__ double s_h[kSumStage];
  __shared__ double sa[kBoostThreads];
  __shared__ double sb[kBoostThreads];
  const int64_t n = n_rows * K;
  double xa = 0.0, xb = 0.0;
  for (int stage = 0; stage < kSumChunk / kSumStage; stage++) {
    const int64_t e0 = blockIdx.x * static_cast<int64_t>(kSumChunk) + static_cast<int64_t>(stage) * kSumStage;
    const int64_t e1 = e0 + kSumStage < n ? e0 + kSumStage : n;
    if (e0 < n) {
      const int64_t r0 = e0 / K, r1 = (e1 + K - 1) / K;
      for (int64_t r = r0 + threadIdx.x; r < r1; r += kBoostThreads) {
        const double w  = weight != nullptr ? weight[r] : 1.0;
        const int label = static_cast<int>(y[r]);
        const double* p = pred + r * K;
        auto emit = [&](int k, double q) {
          double go, ho;
          weigh(k == label ? q + -1.0 : q, q * (1.0 - q), w, lr, &go, &ho);
          const int64_t e = r * K + k;
          g[e]            = go;
          h[e]            = ho;
          if (e >= e0 && e < e1) {
            s_g[e - e0] = go;
            s_h[e - e0] = ho;
          }
        };
        // the same arithmetic, in the same order, as gradient_softmax_rows_kernel
        double top = p[0];
        for (int k = 1; k < K; k++) top = fmax(top, p[k]);
        double div = 0.0;
        for (int k = 0; k < K; k++) div += exp(p[k] - top);
        for (int k = 0; k < K; k++) emit(k, exp(p[k] - top) / div);
      }
    }
    __syncthreads();
    for (int j = 0; j < kSumStage / kBoostThreads; j++) {
      const int64_t e = e0 + threadIdx.x + static_cast<int64_t>(kBoostThreads) * j;
      if (e < e1) {
        xa += fabs(s_g[e - e0]);
        xb += fabs(s_h[e - e0]);
      }
    }
    __syncthreads();
  }
  store_chunk_sums(xa, xb, sa, sb, sum_g, sum_h);
}

__global__ void __launch_bounds__(kBoostThreads)
  add_leaf_values_kernel(const double* __restrict__ leaf, int n_nodes, const int32_t* __restrict__ row_leaf,
                         int64_t n, int K, double* pred)
{
  const int64_t i = blockIdx.x * static_cast<int64_t>(kBoostThreads) + threadIdx.x;
  if (i >= n) return;
  const int64_t r = K == 1 ? i : i / K;
  const int k     = K == 1 ? 0 : static_cast<int>(i - r * K);
  const int node  = row_leaf[r];
  // a row_leaf entry outside the tree is a caller error; such a row keeps its prediction
  if (node >= 0 && node < n_nodes) pred[i] += leaf[static_cast<int64_t>(node) * K + k];
}

template <typename T>
__global__ void __launch_bounds__(kBoostThreads)
  gather_rows_kernel(const T* __restrict__ X, int64_t row_offset, int64_t n_rows, int F,
                     const int64_t* __restrict__ rows, int64_t n, T* __restrict__ out)
{
  const int64_t idx = blockIdx.x * static_cast<int64_t>(kBoostThreads) + threadIdx.x;
  if (idx >= n) return;
  const int64_t i   = idx / F;
  const int j       = static_cast<int>(idx - i * F);
  const int64_t row = rows[i] - row_offset;
  out[idx]          = (row >= 0 && row < n_rows) ? X[row * F + j] : T(0);
}

// Class probabilities from the trees' sums and the initial prediction (legateboost/legateboost.py:507-529 with
// objectives.py:489-531): one read of the sums, one write, where operator by operator the rows are read and written six times
// (500,003 x 8: 93 us in five launches, now 14.5).
// One output: (1 - p, p), a row per thread.
__global__ void __launch_bounds__(kBoostThreads)
  two_class_probabilities_kernel(const double* __restrict__ raw, const double* __restrict__ init, int64_t n, double* __restrict__ out)
{
  const int64_t i = blockIdx.x * static_cast<int64_t>(kBoostThreads) + threadIdx.x;
  if (i >= n) return;
  const double p = 1.0 / (1.0 + exp(-(init[0] + raw[i])));
  reinterpret_cast<double2*>(out)[i] = make_double2(1.0 - p, p);
}

// One row per thread, its entries through the LDS so that memory is read and written in order (a row per lane straight
// from memory is a stride of K doubles between lanes).
template <int kCols>
__global__ void __launch_bounds__(kBoostThreads)
  class_probabilities_kernel(const double* __restrict__ raw, const double* __restrict__ init, int64_t n_rows, double* __restrict__ out)
{
  constexpr int kPitch = kCols | 1;  // rows begin in different banks
  __shared__ double s_v[kBoostThreads * kPitch];
  const int64_t first = blockIdx.x * static_cast<int64_t>(kBoostThreads) * kCols, n = n_rows * kCols;
#pragma unroll
  for (int j = 0; j < kCols; j++) {
    const int e = threadIdx.x + j * kBoostThreads, row = e / kCols, k = e - row * kCols;
    if (first + e < n) s_v[row * kPitch + k] = init[k] + raw[first + e];
  }
  __syncthreads();
  double* const v = s_v + threadIdx.x * kPitch;
  if (blockIdx.x * static_cast<int64_t>(kBoostThreads) + threadIdx.x < n_rows) {
    double e[kCols], top = v[0], div = 0.0;
#pragma unroll
    for (int k = 0; k < kCols; k++) {
      e[k] = v[k];
      top  = fmax(top, e[k]);
    }
#pragma unroll
    for (int k = 0; k < kCols; k++) {
      e[k] = exp(e[k] - top);
      div += e[k];
    }
#pragma unroll
    for (int k = 0; k < kCols; k++) v[k] = e[k] / div;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kCols; j++) {
    const int e = threadIdx.x + j * kBoostThreads, row = e / kCols, k = e - row * kCols;
    if (first + e < n) out[first + e] = s_v[row * kPitch + k];
  }
}

// Any other number of outputs: kLanes lanes of a wave share a row and hold kItems entries each (K <= kLanes * kItems), lane l the entries
// l, l + kLanes, ...: the rows of a wave are one run of memory. kItems = 0: a wave takes a row and goes through it three times. predict_proba
// of 300,000 rows and 3 trees, us, with a row per lane straight from memory, by operators, and now: 12 classes 164, 108, 47; 20 364, 170,
// 69; 100 2207, 809, 340.
template <int kLanes, int kItems>
__global__ void __launch_bounds__(kBoostThreads)
  shared_class_probabilities_kernel(const double* __restrict__ raw, const double* __restrict__ init, int64_t n_rows, int K, double* __restrict__ out)
{
  const int lane  = static_cast<int>(threadIdx.x) % kLanes;
  const int64_t r = blockIdx.x * static_cast<int64_t>(kBoostThreads / kLanes) + threadIdx.x / kLanes;
  if (r >= n_rows) return;  // (all lanes of the row)
  const double* const p = raw + r * K;
  double* const o       = out + r * K;
  auto of_row = [](double v, auto join) {
#pragma unroll
    for (int off = kLanes / 2; off >= 1; off >>= 1) v = join(v, __shfl_xor(v, off, kLanes));
    return v;
  };
  const auto larger = [](double a, double b) { return fmax(a, b); };
  const auto sum    = [](double a, double b) { return a + b; };
  double top = -std::numeric_limits<double>::infinity(), div = 0.0;
  if constexpr (kItems > 0) {
    double e[kItems];
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      const int k = lane + i * kLanes;
      e[i]        = k < K ? init[k] + p[k] : top;
    }
#pragma unroll
    for (int i = 0; i < kItems; i++) top = fmax(top, e[i]);
    top = of_row(top, larger);
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      e[i] = lane + i * kLanes < K ? exp(e[i] - top) : 0.0;
      div += e[i];
    }
    div = of_row(div, sum);
#pragma unroll
    for (int i = 0; i < kItems; i++)
      if (lane + i * kLanes < K) o[lane + i * kLanes] = e[i] / div;
  } else {
    for (int k = lane; k < K; k += kLanes) top = fmax(top, init[k] + p[k]);
    top = of_row(top, larger);
    for (int k = lane; k < K; k += kLanes) {
      const double e = exp(init[k] + p[k] - top);
      div += e;
      o[k] = e;
    }
    div = of_row(div, sum);
    for (int k = lane; k < K; k += kLanes) o[k] /= div;
  }
}

// The initial prediction (legateboost/objectives.py:131-147 and :489-531).
//
// Squared error: the weighted mean of every output in two launches (10,000,000 rows 30 us, 1,000,000 9; the four of the operators
// 97 and 30). A thread adds the entries of one output (kBoostThreads rounded down to whole
// rows take part), four at a time, a workgroup its threads' in a fixed order, one workgroup the workgroups'.
constexpr int kMeanGroups = 1024;
constexpr int kMeanOutputs = kBoostThreads;  // outputs of a row that the threads of a workgroup share

// s: one double per thread; the sum of the threads t = k, k + K, ... in their order for thread k < K
__device__ inline double sum_of_strided(double mine, int K, int threads, double* s)
{
  if (K == 1) {
    s[threadIdx.x] = mine;
    __syncthreads();
    for (int stride = kBoostThreads / 2; stride >= 1; stride >>= 1) {
      if (static_cast<int>(threadIdx.x) < stride) s[threadIdx.x] += s[threadIdx.x + stride];
      __syncthreads();
    }
    const double sum = s[0];
    __syncthreads();
    return sum;
  }
  s[threadIdx.x] = mine;
  __syncthreads();
  double sum = 0.0;
  if (static_cast<int>(threadIdx.x) < K)
    for (int t = threadIdx.x; t < threads; t += K) sum += s[t];
  __syncthreads();
  return sum;
}

// partial: [K + 1][kMeanGroups], the last one of the weights
__global__ void __launch_bounds__(kBoostThreads)
  weighted_sums_kernel(const double* __restrict__ y, const double* __restrict__ weight, int64_t n_rows, int K,
                       double* __restrict__ partial)
{
  __shared__ double s[kBoostThreads];
  const int rows = kBoostThreads / K, threads = rows * K;  // of a step
  const int64_t step = static_cast<int64_t>(gridDim.x) * rows;
  const int row_of = static_cast<int>(threadIdx.x) / K;
  double sum[4] = {}, w_sum[4] = {};
  if (static_cast<int>(threadIdx.x) < threads) {
    for (int64_t r = blockIdx.x * static_cast<int64_t>(rows) + row_of; r < n_rows; r += 4 * step) {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int64_t row = r + u * step;
        if (row < n_rows) {
          const double w = weight != nullptr ? weight[row] : 1.0;
          sum[u] += y[row * K + (static_cast<int>(threadIdx.x) - row_of * K)] * w;
          w_sum[u] += w;
        }
      }
    }
  }
  const double mine   = sum_of_strided((sum[0] + sum[1]) + (sum[2] + sum[3]), K, threads, s);
  const double weights = sum_of_strided((w_sum[0] + w_sum[1]) + (w_sum[2] + w_sum[3]), K, threads, s);
  if (static_cast<int>(threadIdx.x) < K) partial[static_cast<int64_t>(threadIdx.x) * kMeanGroups + blockIdx.x] = mine;
  if (threadIdx.x == 0) partial[static_cast<int64_t>(K) * kMeanGroups + blockIdx.x] = weights;
}

// One workgroup per output
__global__ void __launch_bounds__(kBoostThreads)
  weighted_mean_kernel(const double* __restrict__ partial, int groups, int K, double* __restrict__ mean)
{
  __shared__ double s[kBoostThreads];
  double sum = 0.0, w_sum = 0.0;
  for (int i = threadIdx.x; i < groups; i += kBoostThreads) {
    sum += partial[static_cast<int64_t>(blockIdx.x) * kMeanGroups + i];
    w_sum += partial[static_cast<int64_t>(K) * kMeanGroups + i];
  }
  sum   = sum_of_strided(sum, 1, kBoostThreads, s);
  w_sum = sum_of_strided(w_sum, 1, kBoostThreads, s);
  if (threadIdx.x == 0) mean[blockIdx.x] = sum / w_sum;
}

// Log loss: how often every class occurs, what the labels are and the largest one in one pass that the host waits for once
// (250,007 rows, two classes: 9 us; eight launches and two waits by operators). stats: [0] entries that are no whole number of 0 or more, [1] the largest label,
// [2] entries that are kLabelMost or more, [3 ..] the classes' counts; all zero before.
constexpr int kLabelMost   = 256;
constexpr int kLabelCopies = 4;  // of the LDS counters: one per wave
__global__ void __launch_bounds__(kBoostThreads)
  label_counts_kernel(const double* __restrict__ y, int64_t n, unsigned long long* __restrict__ stats)
{
  __shared__ unsigned s_count[kLabelCopies][kLabelMost];
  __shared__ unsigned s_bad, s_wide, s_most;
  for (int i = threadIdx.x; i < kLabelCopies * kLabelMost; i += kBoostThreads) (&s_count[0][0])[i] = 0;
  if (threadIdx.x == 0) s_bad = s_wide = s_most = 0;
  __syncthreads();
  unsigned* const count = s_count[threadIdx.x >> 6];
  const int64_t step    = static_cast<int64_t>(gridDim.x) * kBoostThreads;
  unsigned bad = 0, wide = 0, zeros = 0, ones = 0;
#pragma unroll 4
  for (int64_t i = blockIdx.x * static_cast<int64_t>(kBoostThreads) + threadIdx.x; i < n; i += step) {
    const double v = y[i];
    if (!(v == floor(v) && v >= 0)) {
      bad++;
    } else if (!(v < kLabelMost)) {
      wide++;
    } else if (v == 0.0) {
      zeros++;  // (the two classes of most data: no lane waits for another one's add)
    } else if (v == 1.0) {
      ones++;
    } else {
      atomicAdd(count + static_cast<int>(v), 1u);
    }
  }
  if (bad != 0) atomicAdd(&s_bad, bad);
  if (wide != 0) atomicAdd(&s_wide, wide);
  if (zeros != 0) atomicAdd(count, zeros);
  if (ones != 0) atomicAdd(count + 1, ones);
  __syncthreads();
  for (int c = threadIdx.x; c < kLabelMost; c += kBoostThreads) {
    unsigned long long all = 0;
    for (int w = 0; w < kLabelCopies; w++) all += s_count[w][c];
    if (all != 0) {
      atomicAdd(stats + 3 + c, all);
      atomicMax(&s_most, static_cast<unsigned>(c));
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    // (once a workgroup: all of them at one address are waited for one after the other)
    if (s_most != 0) atomicMax(stats + 1, static_cast<unsigned long long>(s_most));
    if (s_bad != 0) atomicAdd(stats, static_cast<unsigned long long>(s_bad));
    if (s_wide != 0) atomicAdd(stats + 2, static_cast<unsigned long long>(s_wide));
  }
}

// Two classes: the log odds of class 1; more: the logs of their shares
__global__ void label_priors_kernel(const unsigned long long* __restrict__ stats, int64_t n, int n_outputs, double* __restrict__ init)
{
  const int k = threadIdx.x;
  if (k >= n_outputs) return;
  const double share = static_cast<double>(stats[3 + (n_outputs == 1 ? 1 : k)]) / static_cast<double>(n);
  init[k] = n_outputs == 1 ? -log(1.0 / share - 1.0) : log(share);
}

// Rows that a round leaves out (legateboost/legateboost.py:215-222), one launch for four (250,007 rows: 3.5 us, 14): g and h of a row whose draw is not below `limit`, times 0.
__global__ void __launch_bounds__(kBoostThreads)
  keep_rows_kernel(const double* __restrict__ draw, double limit, int64_t n, int K, double* __restrict__ g, double* __restrict__ h)
{
  const int64_t i = blockIdx.x * static_cast<int64_t>(kBoostThreads) + threadIdx.x;
  if (i >= n || draw[K == 1 ? i : i / K] < limit) return;
  g[i] *= 0.0;
  h[i] *= 0.0;
}

// Bits by value: a copy from the host would have the host wait for all that is queued (memory that is not pinned), or the stream for another
// engine.
struct MaskBits {
  uint32_t words[kMaskFeatures / 32];
};
__global__ void __launch_bounds__(kBoostThreads) feature_mask_kernel(MaskBits bits, int n, uint8_t* mask)
{
  const int i = blockIdx.x * kBoostThreads + threadIdx.x;
  if (i < n) mask[i] = static_cast<uint8_t>(bits.words[i >> 5] >> (i & 31) & 1u);
}

inline unsigned grid_for(int64_t n) { return static_cast<unsigned>((n + kBoostThreads - 1) / kBoostThreads); }

}  // namespace lbt

extern "C" {

int64_t lbt_abs_sum_chunks(int64_t n_rows, int32_t n_outputs)
{
  if (n_rows < 1 || n_outputs < 1) return 0;
  return (n_rows * n_outputs + lbt::kSumChunk - 1) / lbt::kSumChunk;
}

// Gradients at pred, after the leaf values of `add` were added to it; chunk sums of |g| and |h| where `sums` is not null.
static int form_gradients(hipStream_t s, int32_t objective, const lbt::LeafAdd& add, double* pred, const double* y, const double* sample_weight,
                          double learning_rate, int64_t n_rows, int32_t n_outputs, double* g, double* h, double* abs_sum_chunks)
{
  const int64_t n = n_rows * n_outputs;
  const int64_t m = lbt_abs_sum_chunks(n_rows, n_outputs);
  double* sum_g = abs_sum_chunks;
  double* sum_h = abs_sum_chunks != nullptr ? abs_sum_chunks + m : nullptr;
  const bool elementwise = objective == LBT_OBJ_SQUARED_ERROR || n_outputs == 1;
  if (add.leaf != nullptr && !elementwise) {
    // a row's maximum needs all of its predictions
    lbt::ProfScope ps(LBT_PROF_OTHER, s, static_cast<double>(n) * 16.0 + static_cast<double>(n_rows) * 4.0);
    lbt::add_leaf_values_kernel<<<lbt::grid_for(n), lbt::kBoostThreads, 0, s>>>(add.leaf, add.n_nodes, add.row_leaf, n, n_outputs, pred);
  }
  lbt::ProfScope ps(LBT_PROF_OTHER, s, static_cast<double>(n) * (add.leaf != nullptr && elementwise ? 44.0 : 32.0));
  if (elementwise) {
    auto run = [&](auto logistic, auto adds) {
      constexpr bool kLogistic = decltype(logistic)::value, kAdds = decltype(adds)::value;
      if (abs_sum_chunks != nullptr)
        lbt::gradient_elementwise_sums_kernel<kLogistic, kAdds><<<static_cast<unsigned>(m), lbt::kBoostThreads, 0, s>>>(
          add, pred, y, sample_weight, learning_rate, n, n_outputs, g, h, sum_g, sum_h);
      else
        lbt::gradient_elementwise_kernel<kLogistic, kAdds><<<lbt::grid_for(n), lbt::kBoostThreads, 0, s>>>(
          add, pred, y, sample_weight, learning_rate, n, n_outputs, g, h);
    };
    auto with = [&](auto logistic) { add.leaf != nullptr ? run(logistic, std::true_type{}) : run(logistic, std::false_type{}); };
    objective == LBT_OBJ_SQUARED_ERROR ? with(std::false_type{}) : with(std::true_type{});
  } else if (abs_sum_chunks != nullptr) {
    if (n_outputs <= lbt::kSoftmaxCols)
      lbt::gradient_softmax_kernel<true><<<static_cast<unsigned>(m), lbt::kBoostThreads, 0, s>>>(pred, y, sample_weight, learning_rate, n_rows,
                                                                                                 n_outputs, g, h, sum_g, sum_h);
    else
      lbt::gradient_softmax_rows_sums_kernel<<<static_cast<unsigned>(m), lbt::kBoostThreads, 0, s>>>(pred, y, sample_weight, learning_rate, n_rows,
                                                                                                     n_outputs, g, h, sum_g, sum_h);
  } else if (lbt::softmax_by_entry(n, n_outputs)) {
    const unsigned grid = static_cast<unsigned>((n + lbt::kSumStage - 1) / lbt::kSumStage);
    lbt::gradient_softmax_kernel<false><<<grid, lbt::kBoostThreads, 0, s>>>(pred, y, sample_weight, learning_rate, n_rows, n_outputs, g, h,
                                                                            nullptr, nullptr);
  } else {
    const unsigned grid = lbt::grid_for(n_rows);
#define LBT_SOFTMAX(C)                                                                                                      \
  lbt::gradient_softmax_rows_kernel<C><<<grid, lbt::kBoostThreads, 0, s>>>(pred, y, sample_weight, learning_rate, n_rows, \
                                                                           n_outputs, g, h)
    switch (n_outputs) {
      case 2: LBT_SOFTMAX(2); break;
      case 3: LBT_SOFTMAX(3); break;
      case 4: LBT_SOFTMAX(4); break;
      case 5: LBT_SOFTMAX(5); break;
      case 6: LBT_SOFTMAX(6); break;
      case 7: LBT_SOFTMAX(7); break;
      case 8: LBT_SOFTMAX(8); break;
      case 10: LBT_SOFTMAX(10); break;
      case 16: LBT_SOFTMAX(16); break;
      default: LBT_SOFTMAX(0); break;
    }
#undef LBT_SOFTMAX
  }
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

// What the three calls ask of their arguments.
static int check_gradients(const double* pred, const double* y, int64_t n_rows, int32_t n_outputs, const double* g, const double* h,
                           const double* abs_sum_chunks)
{
  LBT_REQUIRE(pred && y && g && h, "null pointer");
  LBT_REQUIRE(g != pred && h != pred && g != y && h != y && g != h, "outputs may not alias the inputs or each other");
  if (abs_sum_chunks == nullptr) return LBT_OK;
  // the chunk sums are written while the pass still reads pred and y and writes g and h
  const char* c0 = reinterpret_cast<const char*>(abs_sum_chunks);
  const char* c1 = c0 + 2 * sizeof(double) * static_cast<size_t>(lbt_abs_sum_chunks(n_rows, n_outputs));
  const size_t bytes = sizeof(double) * static_cast<size_t>(n_rows * n_outputs);
  for (const double* a : {pred, g, h}) {
    const char* a0 = reinterpret_cast<const char*>(a);
    LBT_REQUIRE(c1 <= a0 || a0 + bytes <= c0, "abs_sum_chunks may not alias pred, g or h");
  }
  const char* y0 = reinterpret_cast<const char*>(y);  // at least n_rows labels
  LBT_REQUIRE(c1 <= y0 || y0 + sizeof(double) * static_cast<size_t>(n_rows) <= c0, "abs_sum_chunks may not alias y");
  return LBT_OK;
}

int lbt_weighted_gradient_sums(void* stream, int32_t objective, const double* pred, const double* y,
                               const double* sample_weight, double learning_rate, int64_t n_rows,
                               int32_t n_outputs, double* g, double* h, double* abs_sum_chunks)
{
  LBT_REQUIRE(objective == LBT_OBJ_SQUARED_ERROR || objective == LBT_OBJ_LOG_LOSS, "unknown objective %d", objective);
  LBT_REQUIRE(n_rows >= 1 && n_outputs >= 1, "bad shape");
  LBT_REQUIRE(n_rows * n_outputs < (int64_t(1) << 38), "too many elements");
  LBT_REQUIRE(abs_sum_chunks, "null pointer");
  LBT_TRY(check_gradients(pred, y, n_rows, n_outputs, g, h, abs_sum_chunks));
  // (nothing is added: the predictions are only read)
  return form_gradients(static_cast<hipStream_t>(stream), objective, lbt::LeafAdd{}, const_cast<double*>(pred), y, sample_weight, learning_rate, n_rows,
                        n_outputs, g, h, abs_sum_chunks);
}

int lbt_weighted_gradient(void* stream, int32_t objective, const double* pred, const double* y,
                          const double* sample_weight, double learning_rate, int64_t n_rows,
                          int32_t n_outputs, double* g, double* h)
{
  LBT_REQUIRE(objective == LBT_OBJ_SQUARED_ERROR || objective == LBT_OBJ_LOG_LOSS, "unknown objective %d", objective);
  LBT_REQUIRE(n_rows >= 0 && n_outputs >= 1, "bad shape");
  LBT_REQUIRE(n_rows * n_outputs < (int64_t(1) << 38), "too many elements");
  if (n_rows == 0) return LBT_OK;
  LBT_TRY(check_gradients(pred, y, n_rows, n_outputs, g, h, nullptr));
  return form_gradients(static_cast<hipStream_t>(stream), objective, lbt::LeafAdd{}, const_cast<double*>(pred), y, sample_weight, learning_rate, n_rows,
                        n_outputs, g, h, nullptr);
}

int lbt_next_gradient(void* stream, int32_t objective, const double* leaf_value, int32_t n_nodes, const int32_t* row_leaf, double* pred,
                      const double* y, const double* sample_weight, double learning_rate, int64_t n_rows, int32_t n_outputs, double* g,
                      double* h, double* abs_sum_chunks)
{
  LBT_REQUIRE(objective == LBT_OBJ_SQUARED_ERROR || objective == LBT_OBJ_LOG_LOSS, "unknown objective %d", objective);
  LBT_REQUIRE(n_rows >= 0 && n_outputs >= 1 && n_nodes >= 1, "bad shape");
  LBT_REQUIRE(n_rows * n_outputs < (int64_t(1) << 38), "too many elements");
  if (n_rows == 0) return LBT_OK;
  LBT_REQUIRE(leaf_value && row_leaf, "null pointer");
  LBT_TRY(check_gradients(pred, y, n_rows, n_outputs, g, h, abs_sum_chunks));
  // the predictions are written while everything else is read: none of what is written may overlap what is read, or one another
  struct Range {
    const void* begin;
    int64_t bytes;
  };
  const int64_t real = sizeof(double), all = real * n_rows * n_outputs, labels = objective == LBT_OBJ_LOG_LOSS && n_outputs > 1 ? real * n_rows : all;
  const Range ranges[] = {{pred, all}, {g, all}, {h, all}, {abs_sum_chunks, 2 * real * lbt_abs_sum_chunks(n_rows, n_outputs)},
                          {leaf_value, real * n_nodes * n_outputs}, {row_leaf, static_cast<int64_t>(sizeof(int32_t)) * n_rows}, {y, labels},
                          {sample_weight, real * n_rows}};
  constexpr int kWritten = 4;
  for (int i = 0; i < kWritten; i++)
    for (const Range* other = ranges + i + 1; other != std::end(ranges); other++) {
      const char *a = static_cast<const char*>(ranges[i].begin), *b = static_cast<const char*>(other->begin);
      LBT_REQUIRE(a == nullptr || b == nullptr || a + ranges[i].bytes <= b || b + other->bytes <= a, "outputs may not alias the inputs or each other");
    }
  return form_gradients(static_cast<hipStream_t>(stream), objective, lbt::LeafAdd{leaf_value, n_nodes, row_leaf}, pred, y, sample_weight, learning_rate,
                        n_rows, n_outputs, g, h, abs_sum_chunks);
}

size_t lbt_weighted_mean_workspace_bytes(int32_t n_outputs)
{
  if (n_outputs < 1 || n_outputs > lbt::kMeanOutputs) return 0;
  return sizeof(double) * static_cast<size_t>(n_outputs + 1) * lbt::kMeanGroups;
}

int lbt_weighted_mean(void* stream, const double* y, const double* sample_weight, int64_t n_rows, int32_t n_outputs,
                      double* mean, void* workspace, size_t workspace_bytes)
{
  LBT_REQUIRE(n_rows >= 1 && n_outputs >= 1 && n_outputs <= lbt::kMeanOutputs, "bad shape");
  LBT_REQUIRE(n_rows * n_outputs < (int64_t(1) << 38), "too many elements");
  LBT_REQUIRE(y && mean && workspace, "null pointer");
  LBT_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 8 == 0, "workspace must be 8-byte aligned");
  if (workspace_bytes < lbt_weighted_mean_workspace_bytes(n_outputs)) {
    lbt::set_error("workspace too small");
    return LBT_ERR_WORKSPACE;
  }
  hipStream_t s      = static_cast<hipStream_t>(stream);
  const int64_t rows = lbt::kBoostThreads / n_outputs;
  const int groups   = static_cast<int>(std::min<int64_t>((n_rows + 4 * rows - 1) / (4 * rows), lbt::kMeanGroups));
  double* partial    = static_cast<double*>(workspace);
  lbt::ProfScope ps(LBT_PROF_OTHER, s, static_cast<double>(n_rows) * n_outputs * 8.0);
  lbt::weighted_sums_kernel<<<groups, lbt::kBoostThreads, 0, s>>>(y, sample_weight, n_rows, n_outputs, partial);
  lbt::weighted_mean_kernel<<<n_outputs, lbt::kBoostThreads, 0, s>>>(partial, groups, n_outputs, mean);
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

int lbt_label_counts(void* stream, const double* y, int64_t n, int64_t* stats)
{
  LBT_REQUIRE(n >= 1 && n < (int64_t(1) << 38), "bad shape");
  LBT_REQUIRE(y && stats, "null pointer");
  hipStream_t s    = static_cast<hipStream_t>(stream);
  const int groups = static_cast<int>(std::min<int64_t>((n + 8 * lbt::kBoostThreads - 1) / (8 * lbt::kBoostThreads), 1024));
  lbt::ProfScope ps(LBT_PROF_OTHER, s, static_cast<double>(n) * 8.0);
  lbt::label_counts_kernel<<<groups, lbt::kBoostThreads, 0, s>>>(y, n, reinterpret_cast<unsigned long long*>(stats));
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

int lbt_label_priors(void* stream, const int64_t* stats, int64_t n, int32_t n_outputs, double* init)
{
  LBT_REQUIRE(n >= 1 && n_outputs >= 1 && n_outputs <= lbt::kLabelMost, "bad shape");
  LBT_REQUIRE(stats && init, "null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  lbt::ProfScope ps(LBT_PROF_OTHER, s);
  lbt::label_priors_kernel<<<1, lbt::kLabelMost, 0, s>>>(reinterpret_cast<const unsigned long long*>(stats), n, n_outputs, init);
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

int lbt_keep_rows(void* stream, const double* draw, double limit, int64_t n_rows, int32_t n_outputs, double* g, double* h)
{
  LBT_REQUIRE(n_rows >= 0 && n_outputs >= 1, "bad shape");
  LBT_REQUIRE(n_rows * n_outputs < (int64_t(1) << 38), "too many elements");
  if (n_rows == 0) return LBT_OK;
  LBT_REQUIRE(draw && g && h, "null pointer");
  LBT_REQUIRE(g != h && draw != g && draw != h, "the arrays may not alias each other");
  hipStream_t s   = static_cast<hipStream_t>(stream);
  const int64_t n = n_rows * n_outputs;
  lbt::ProfScope ps(LBT_PROF_OTHER, s, static_cast<double>(n) * 8.0);
  lbt::keep_rows_kernel<<<lbt::grid_for(n), lbt::kBoostThreads, 0, s>>>(draw, limit, n, n_outputs, g, h);
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

int lbt_feature_mask(void* stream, const uint8_t* host_mask, int32_t n_features, uint8_t* feature_set)
{
  LBT_REQUIRE(n_features >= 0, "bad shape");
  if (n_features == 0) return LBT_OK;
  LBT_REQUIRE(host_mask && feature_set, "null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  lbt::ProfScope ps(LBT_PROF_OTHER, s, static_cast<double>(n_features));
  for (int32_t first = 0; first < n_features; first += lbt::kMaskFeatures) {
    const int n = std::min(lbt::kMaskFeatures, n_features - first);
    lbt::MaskBits bits{};
    for (int i = 0; i < n; i++)
      if (host_mask[first + i] != 0) bits.words[i >> 5] |= 1u << (i & 31);
    lbt::feature_mask_kernel<<<lbt::grid_for(n), lbt::kBoostThreads, 0, s>>>(bits, n, feature_set + first);
  }
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

int lbt_class_probabilities(void* stream, const double* raw, const double* init, int64_t n_rows, int32_t n_outputs, double* out)
{
  LBT_REQUIRE(n_rows >= 0 && n_outputs >= 1, "bad shape");
  LBT_REQUIRE(n_rows * n_outputs < (int64_t(1) << 38), "too many elements");
  if (n_rows == 0) return LBT_OK;
  LBT_REQUIRE(raw && init && out, "null pointer");
  hipStream_t s     = static_cast<hipStream_t>(stream);
  const int64_t n   = n_rows * n_outputs;
  const bool binary = n_outputs == 1;
  LBT_REQUIRE(raw != out, "the output may not alias the input");
  LBT_REQUIRE(!binary || reinterpret_cast<uintptr_t>(out) % 16 == 0, "the output must be 16-byte aligned: a row's two probabilities are stored together");
  lbt::ProfScope ps(LBT_PROF_OTHER, s, static_cast<double>(n) * (binary ? 24.0 : 16.0));
  if (binary) {
    lbt::two_class_probabilities_kernel<<<lbt::grid_for(n), lbt::kBoostThreads, 0, s>>>(raw, init, n, out);
  } else {
    auto shared = [&](auto lanes_c, auto items_c) {
      constexpr int kLanes = decltype(lanes_c)::value, kItems = decltype(items_c)::value, kRows = lbt::kBoostThreads / kLanes;
      lbt::shared_class_probabilities_kernel<kLanes, kItems>
        <<<static_cast<unsigned>((n_rows + kRows - 1) / kRows), lbt::kBoostThreads, 0, s>>>(raw, init, n_rows, n_outputs, out);
    };
    using std::integral_constant;
#define LBT_SOFTMAX(C) lbt::class_probabilities_kernel<C><<<lbt::grid_for(n_rows), lbt::kBoostThreads, 0, s>>>(raw, init, n_rows, out)
    switch (n_outputs) {
      case 2: LBT_SOFTMAX(2); break;
      case 3: LBT_SOFTMAX(3); break;
      case 4: LBT_SOFTMAX(4); break;
      case 5: LBT_SOFTMAX(5); break;
      case 6: LBT_SOFTMAX(6); break;
      case 7: LBT_SOFTMAX(7); break;
      case 8: LBT_SOFTMAX(8); break;
      case 10: LBT_SOFTMAX(10); break;
      case 16: LBT_SOFTMAX(16); break;
      default:
        if (n_outputs <= 12) shared(integral_constant<int, 4>{}, integral_constant<int, 3>{});
        else if (n_outputs <= 16) shared(integral_constant<int, 4>{}, integral_constant<int, 4>{});
        else if (n_outputs <= 24) shared(integral_constant<int, 8>{}, integral_constant<int, 3>{});
        else if (n_outputs <= 32) shared(integral_constant<int, 8>{}, integral_constant<int, 4>{});
        else if (n_outputs <= 48) shared(integral_constant<int, 16>{}, integral_constant<int, 3>{});
        else if (n_outputs <= 64) shared(integral_constant<int, 16>{}, integral_constant<int, 4>{});
        else if (n_outputs <= 128) shared(integral_constant<int, 32>{}, integral_constant<int, 4>{});
        else if (n_outputs <= 256) shared(integral_constant<int, 64>{}, integral_constant<int, 4>{});
        else shared(integral_constant<int, 64>{}, integral_constant<int, 0>{});
        break;
    }
#undef LBT_SOFTMAX
  }
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

int lbt_add_leaf_values(void* stream, const double* leaf_value, int32_t n_nodes,
                        const int32_t* row_leaf, int64_t n_rows, int32_t n_outputs, double* pred)
{
  LBT_REQUIRE(n_rows >= 0 && n_outputs >= 1 && n_nodes >= 1, "bad shape");
  LBT_REQUIRE(n_rows * n_outputs < (int64_t(1) << 38), "too many elements");
  if (n_rows == 0) return LBT_OK;
  LBT_REQUIRE(leaf_value && row_leaf && pred, "null pointer");
  hipStream_t s   = static_cast<hipStream_t>(stream);
  const int64_t n = n_rows * n_outputs;
  lbt::ProfScope ps(LBT_PROF_OTHER, s, static_cast<double>(n) * 16.0 + static_cast<double>(n_rows) * 4.0);
  lbt::add_leaf_values_kernel<<<lbt::grid_for(n), lbt::kBoostThreads, 0, s>>>(leaf_value, n_nodes, row_leaf, n,
                                                                              n_outputs, pred);
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

int lbt_gather_rows(void* stream, const void* X, int32_t x_dtype, int64_t row_offset, int64_t n_rows,
                    int32_t n_features, const int64_t* sample_rows, int64_t n_samples,
                    int32_t samples_on_host, int64_t* staging, void* out)
{
  LBT_REQUIRE(x_dtype == LBT_F32 || x_dtype == LBT_F64, "unsupported X dtype %d", x_dtype);
  LBT_REQUIRE(n_rows >= 0 && n_features >= 1 && n_samples >= 0, "bad shape");
  LBT_REQUIRE(n_samples * n_features < (int64_t(1) << 38), "too many elements");
  if (n_samples == 0) return LBT_OK;
  LBT_REQUIRE(sample_rows && out, "null pointer");
  LBT_REQUIRE(n_rows == 0 || X, "null X");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t* rows = sample_rows;
  if (samples_on_host) {
    LBT_REQUIRE(staging != nullptr, "staging buffer needed for host sample rows");
    LBT_HIP(hipMemcpyAsync(staging, sample_rows, sizeof(int64_t) * n_samples, hipMemcpyHostToDevice, s));
    rows = staging;
  }
  const int64_t n = n_samples * n_features;
  lbt::ProfScope ps(LBT_PROF_OTHER, s);
  if (x_dtype == LBT_F32)
    lbt::gather_rows_kernel<float><<<lbt::grid_for(n), lbt::kBoostThreads, 0, s>>>(
      static_cast<const float*>(X), row_offset, n_rows, n_features, rows, n, static_cast<float*>(out));
  else
    lbt::gather_rows_kernel<double><<<lbt::grid_for(n), lbt::kBoostThreads, 0, s>>>(
      static_cast<const double*>(X), row_offset, n_rows, n_features, rows, n, static_cast<double*>(out));
  LBT_HIP(hipGetLastError());
  return LBT_OK;
}

}  // extern "C"
