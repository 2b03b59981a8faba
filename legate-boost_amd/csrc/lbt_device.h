// Device functions shared by the two tree builders (lbt_build_tree.hip, lbt_small_tree.hip).
#pragma once

#include "lbt_internal.h"

namespace lbt {

template <typename T>
struct KeyOf;
template <>
struct KeyOf<float> {
  using type = uint32_t;
};
template <>
struct KeyOf<double> {
  using type = uint64_t;
};

// Order-preserving map from IEEE bits to unsigned integers (-0.0 < +0.0).
__device__ inline uint32_t to_key(float v)
{
  uint32_t u = __float_as_uint(v);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ inline uint64_t to_key(double v)
{
  uint64_t u = static_cast<uint64_t>(__double_as_longlong(v));
  return (u & 0x8000000000000000ULL) ? ~u : (u | 0x8000000000000000ULL);
}
__device__ inline float from_key(uint32_t k)
{
  uint32_t u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
  return __uint_as_float(u);
}
__device__ inline double from_key(uint64_t k)
{
  uint64_t u = (k & 0x8000000000000000ULL) ? (k & 0x7fffffffffffffffULL) : ~k;
  return __longlong_as_double(static_cast<long long>(u));
}

// Running sums over the 64 lanes of a wave through the lanes' own data paths (DPP operands)
// instead of LDS permutes, of which a 64-bit scan by shuffles needs two dozen: inside every row
// of 16 lanes by shifts of 1, 2, 4 and 8 lanes (a lane without a source reads zero), then the
// last lane of row 0 into row 1 and of row 2 into row 3, then lane 31 into rows 2 and 3.
// All 64 lanes must be active.
template <int kCtrl, int kRowMask>
__device__ __forceinline__ int64_t dpp_take(int64_t v)
{
  const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(static_cast<uint32_t>(v)), kCtrl, kRowMask, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(v >> 32), kCtrl, kRowMask, 0xf, true);
  return static_cast<int64_t>((static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) | static_cast<uint32_t>(lo));
}
__device__ __forceinline__ int64_t wave_inclusive_sum(int64_t v)
{
  v += dpp_take<0x111, 0xf>(v);  // row_shr:1
  v += dpp_take<0x112, 0xf>(v);  // row_shr:2
  v += dpp_take<0x114, 0xf>(v);  // row_shr:4
  v += dpp_take<0x118, 0xf>(v);  // row_shr:8
  v += dpp_take<0x142, 0xa>(v);  // row_bcast:15, rows 1 and 3
  v += dpp_take<0x143, 0xc>(v);  // row_bcast:31, rows 2 and 3
  return v;
}
// value of lane `src` (the same for the whole wave) in every lane
__device__ __forceinline__ int64_t wave_read_lane(int64_t v, int src)
{
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(static_cast<uint32_t>(v)), src));
  const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v >> 32), src));
  return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}

struct Cand {
  double gain;
  int bin;
};

// Total order equivalent to the reference's 512 strided threads followed by a
// rank-ordered reduction with op(a,b) = a.gain > b.gain ? a : b: larger gain
// wins; among equal gains the larger (bin mod 512); inside one residue class
// the smaller bin. Only bins with gain > 0 are candidates.
__device__ inline bool cand_better(const Cand& a, const Cand& b)
{
  if (a.bin < 0) return false;
  if (b.bin < 0) return true;
  if (a.gain != b.gain) return a.gain > b.gain;
  int ra = a.bin & 511, rb = b.bin & 511;
  if (ra != rb) return ra > rb;
  return a.bin < b.bin;
}

__device__ inline void add_gain(double& gain, bool& dead, const I64Pair& ls, const I64Pair& ns, double inv_g,
                                double inv_h, double l1, double reg, double min_split_gain)
{
  const int64_t rg = ns.grad - ls.grad, rh = ns.hess - ls.hess;
  if (dead) return;
  if (ls.hess <= 0 || rh <= 0) {
    // build_tree.cu:727-730: one output without a valid split on this bin voids the bin
    dead = true;
    gain = 0;
    return;
  }
  gain += calculate_gain(static_cast<double>(ls.grad) * inv_g, static_cast<double>(ls.hess) * inv_h,
                         static_cast<double>(rg) * inv_g, static_cast<double>(rh) * inv_h,
                         static_cast<double>(ns.grad) * inv_g, static_cast<double>(ns.hess) * inv_h, l1, reg,
                         min_split_gain);
}

}  // namespace lbt
