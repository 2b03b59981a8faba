// Prediction by ranks (lbt_predict_ranked.hip) as lbt_predict sees it.
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

// Scratch of predict_ranked, or 0 when it would not take the call.
size_t ranked_workspace_bytes(int64_t N, int F, int n_trees, const int32_t* tree_nodes, int K, int x_dtype);

// Sets *done when the call was taken. *overflow: null, or a device word that is not 0 after the launches when a feature
// has more thresholds than there are ranks; nothing was computed then.
template <typename T>
int predict_ranked(hipStream_t stream, const T* X, int64_t N, int F, int n_trees, const double* const* leaf,
                   const int32_t* const* feature, const double* const* split, const int32_t* tree_nodes, int K,
                   double* out, void* workspace, size_t workspace_bytes, bool* done, const int32_t** overflow);

}  // namespace lbt
