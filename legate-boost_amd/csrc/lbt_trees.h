// Trees as the traversals see them, and the prediction by ranks (lbt_predict_ranked.hip) as lbt_predict sees it.
#pragma once

#include "lbt_internal.h"

namespace lbt {

constexpr size_t kRankedChunkBytes = 256u << 20;   // ranks held at a time

// x <= t for a float x holds exactly when x <= (the largest float that is <= t)
__device__ inline float round_down_to_float(double d)
{
  float f = static_cast<float>(d);
  if (static_cast<double>(f) > d) {  // false for NaN
    uint32_t b = __float_as_uint(f);
    if (f > 0.0f)
      b -= 1;
    else if (f == 0.0f)
      b = 0x80000001u;
    else
      b += 1;
    f = __uint_as_float(b);
  }
  return f;
}

// A node of a packed tree: threshold in X's type, feature, index of the right child (the left one lies before it). A leaf is a
// node that always steps to itself (threshold NaN, "right child" = itself), so a walk is a fixed number of identical
// steps to right - (x <= threshold).
template <typename T>
struct PackedNode;
template <>
struct alignas(8) PackedNode<float> {
  float thr;
  uint32_t feat_right;  // byte offset of the feature in a row (4 * feature) in the low half, right child in the high half
};
template <>
struct alignas(16) PackedNode<double> {
  double thr;
  int32_t feat;
  int32_t right;
};
constexpr int kMaxPackedFeatures = 16383;  // a float node holds 4 * feature in 16 bits
constexpr int kMaxPackedNodes    = 65535;  // and the right child

template <typename T>
__device__ inline PackedNode<T> pack_node(int i, int feature, double split, int F, int n_nodes)
{
  // a node whose children would lie past the arrays, or whose feature does not exist, ends the walk
  const bool is_leaf = feature < 0 || feature >= F || 2 * static_cast<int64_t>(i) + 2 >= n_nodes;
  const int right    = is_leaf ? i : 2 * i + 2;
  PackedNode<T> nd;
  if constexpr (sizeof(T) == 4) {
    nd.thr        = is_leaf ? __uint_as_float(0x7fc00000u) : round_down_to_float(split);
    nd.feat_right = (is_leaf ? 0u : static_cast<uint32_t>(feature) * 4u) | (static_cast<uint32_t>(right) << 16);
  } else {
    nd.thr   = is_leaf ? __longlong_as_double(0x7ff8000000000000LL) : split;
    nd.feat  = is_leaf ? 0 : feature;
    nd.right = right;
  }
  return nd;
}
template <typename T>
__device__ __forceinline__ int step_from(const PackedNode<T>& nd, const T* x)
{
  if constexpr (sizeof(T) == 4) {
    const float xv = *reinterpret_cast<const float*>(reinterpret_cast<const unsigned char*>(x) + (nd.feat_right & 0xffffu));
    return static_cast<int>(nd.feat_right >> 16) - (xv <= nd.thr ? 1 : 0);
  } else {
    return nd.right - (x[nd.feat] <= nd.thr ? 1 : 0);
  }
}

// Sums g, h [n_nodes][K] of an update, of which every row's lie at the node it stops in: adds what the children of a node
// that leads on hold to it, deepest level first. One workgroup; the arrays in the LDS or in memory.
__device__ inline void sum_inner_nodes(const int32_t* feature, int n_nodes, int K, double* g, double* h)
{
  int depth = 0;
  while (((int64_t(1) << (depth + 1)) - 1) < n_nodes) depth++;
  for (int d = depth - 1; d >= 0; d--) {
    const int64_t first = (int64_t(1) << d) - 1, count = int64_t(1) << d;
    for (int64_t i = threadIdx.x; i < count * K; i += blockDim.x) {
      const int64_t node = first + i / K;
      const int k        = static_cast<int>(i % K);
      if (node < n_nodes && feature[node] != -1) {
        double gs = 0.0, hs = 0.0;
        if (2 * node + 1 < n_nodes) {
          gs += g[(2 * node + 1) * K + k];
          hs += h[(2 * node + 1) * K + k];
        }
        if (2 * node + 2 < n_nodes) {
          gs += g[(2 * node + 2) * K + k];
          hs += h[(2 * node + 2) * K + k];
        }
        g[node * K + k] += gs;
        h[node * K + k] += hs;
      }
    }
    __syncthreads();
  }
}

// update_tree.cc:104-117
__device__ inline double updated_leaf(double g, double h, double l1, double l2)
{
  return h > 0.0 ? calculate_leaf_value(g, h, l1, l2) : 0.0;
}

// Scratch of predict_ranked, or 0 when it would not take the call.
size_t ranked_workspace_bytes(int64_t N, int F, int n_trees, const int32_t* tree_nodes, int K, int x_dtype);

// Sets *done when the call was taken. *overflow: null, or a device word that is not 0 after the launches when a feature
// has more thresholds than there are ranks; nothing was computed then.
template <typename T>
int predict_ranked(hipStream_t stream, const T* X, int64_t N, int F, int n_trees, const double* const* leaf,
                   const int32_t* const* feature, const double* const* split, const int32_t* tree_nodes, int K,
                   double* out, void* workspace, size_t workspace_bytes, bool* done, const int32_t** overflow);

}  // namespace lbt
