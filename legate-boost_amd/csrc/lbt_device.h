// Device functions shared by the tree builders (lbt_build_tree.hip, lbt_small_tree.hip, lbt_mid_tree.hip, lbt_direct_level.hip).
#pragma once

#include <limits>

#include "lbt_internal.h"

#include <type_traits>

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

__device__ __forceinline__ uint32_t wave_read_lane32(uint32_t v, int src)
{
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), src));
}

__device__ __forceinline__ double wave_read_lane_f64(double v, int src)
{
  return __longlong_as_double(wave_read_lane(static_cast<int64_t>(__double_as_longlong(v)), src));
}

// Values that loads bring, when all of them are here: hipcc moves a load behind the branch that is its only use, where a wave
// then waits for it alone.
__device__ __forceinline__ void arrived(int2& v) { asm volatile("" : "+v"(v.x), "+v"(v.y)); }
__device__ __forceinline__ void arrived(I64Pair& v) { asm volatile("" : "+v"(v.grad), "+v"(v.hess)); }
__device__ __forceinline__ void arrived(uint4& v) { asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w)); }

// put(i, take(i)) for i = threadIdx.x, + kT, ... below n: kAhead loads are under way at once. (A loop over both, as hipcc
// leaves it, waits for every load: 2 us each where another die wrote what it reads.)
template <int kT, int kAhead, typename Take, typename Put>
__device__ __forceinline__ void copy_ahead(int n, Take take, Put put)
{
  for (int i0 = threadIdx.x; i0 < n; i0 += kT * kAhead) {
    decltype(take(0)) v[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; u++) v[u] = take(min(i0 + u * kT, n - 1));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kAhead; u++)
      if (i0 + u * kT < n) put(i0 + u * kT, v[u]);
  }
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

// Inclusive sums over a wave modulo 2^32 (see wave_inclusive_sum): the lower halves of longer sums wrap here
template <int kCtrl, int kRowMask>
__device__ __forceinline__ uint32_t dpp_take32(uint32_t v)
{
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), kCtrl, kRowMask, 0xf, true));
}
__device__ __forceinline__ uint32_t wave_inclusive_sum32(uint32_t v)
{
  v += dpp_take32<0x111, 0xf>(v);
  v += dpp_take32<0x112, 0xf>(v);
  v += dpp_take32<0x114, 0xf>(v);
  v += dpp_take32<0x118, 0xf>(v);
  v += dpp_take32<0x142, 0xa>(v);
  v += dpp_take32<0x143, 0xc>(v);
  return v;
}

// Largest value of a wave, in every lane, in the lanes' own data paths (see wave_inclusive_sum): a maximum of gains by LDS
// permutes is 18 of them one after the other, here 12 operations and more for the ties.
__device__ __forceinline__ unsigned wave_max_u32(unsigned v)
{
  auto take = [&](auto ctrl, auto rows) {
    const unsigned o = static_cast<unsigned>(__builtin_amdgcn_update_dpp(
      0, static_cast<int>(v), decltype(ctrl)::value, decltype(rows)::value, 0xf, true));
    v = o > v ? o : v;
  };
  using std::integral_constant;
  take(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});
  take(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});
  take(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});
  take(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});
  take(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});
  take(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});
  return static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

// The lane that holds the best of a wave's candidates (gain, bin) in the order of cand_better; -1: there is none.
// Candidates have bin >= 0 and a positive gain.
__device__ __forceinline__ int wave_best_lane(double gain, int bin)
{
  const unsigned own_hi = bin >= 0 ? static_cast<unsigned>(__double_as_longlong(gain) >> 32) : 0u;
  const unsigned own_lo = static_cast<unsigned>(__double_as_longlong(gain)), own_rank = static_cast<unsigned>(bin & 511) + 1u;
  const unsigned hi = wave_max_u32(own_hi);
  const unsigned lo = wave_max_u32(bin >= 0 && own_hi == hi ? own_lo : 0u);
  const bool holds  = bin >= 0 && own_hi == hi && own_lo == lo;
  const unsigned rank = wave_max_u32(holds ? own_rank : 0u);
  const unsigned low  = wave_max_u32(holds && own_rank == rank ? ~static_cast<unsigned>(bin) : 0u);
  const unsigned long long who = __ballot(holds && ~static_cast<unsigned>(bin) == low);
  return who != 0 ? __builtin_ctzll(who) : -1;
}

// The largest gain of a wave and, of the lanes that hold it, the largest key.
__device__ __forceinline__ void wave_best_key(double& best, unsigned& key)
{
  // gains are not negative: their bits compare as whole numbers, upper halves first
  const unsigned own_hi = static_cast<unsigned>(__double_as_longlong(best) >> 32);
  const unsigned own_lo = static_cast<unsigned>(__double_as_longlong(best));
  const unsigned hi = wave_max_u32(own_hi);
  const unsigned lo = wave_max_u32(own_hi == hi ? own_lo : 0u);
  key  = wave_max_u32(own_hi == hi && own_lo == lo ? key : 0u);
  best = __longlong_as_double(static_cast<int64_t>(static_cast<unsigned long long>(hi) << 32 | lo));
}

// The same with what belongs to the gain: its feature and the bin in it. Keys of different candidates differ.
__device__ __forceinline__ void wave_best_split(double& gain, unsigned& key, int& ft, int& rel)
{
  const double own_gain  = gain;
  const unsigned own_key = key;
  wave_best_key(gain, key);
  const unsigned long long who = __ballot(key != 0 && own_key == key && own_gain == gain);
  if (who != 0) {
    const int from = __builtin_ctzll(who);
    ft  = __builtin_amdgcn_readlane(ft, from);
    rel = __builtin_amdgcn_readlane(rel, from);
  }
}

// leaf_gain without branches (the lanes of a wave hold both signs), same results
__device__ __forceinline__ double leaf_gain_select(double grad, double hess, double l1, double reg)
{
  const double z = grad > l1 ? grad - l1 : (grad < -l1 ? grad + l1 : 0.0);
  return (z * z) / (hess + reg);
}

// n / d, where neither is near the ends of the exponent's range (quotient_from). It is what `/` does without the scaling and the special
// cases, three instructions of eleven.
__device__ __forceinline__ double quotient_plain(double n, double d) { return quotient_from(n, d, __builtin_amdgcn_rcp(d)); }
// Without l1 the sums of grads are squared as they are. Sums are whole numbers below 2^35 times inv_g (inv_h); a denominator is at
// least reg where its quotient counts.
__device__ __forceinline__ bool plain_quotients(double l1, double inv_g, double inv_h, double reg)
{
  auto ordinary = [](double v) { return v >= 1e-60 && v <= 1e60; };
  return l1 == 0.0 && ordinary(inv_g) && ordinary(inv_h) && ordinary(reg);
}

// Sum of the threads before this one; all threads of the workgroup call it. s_wave: one int per wave.
template <int kT>
__device__ __forceinline__ int block_exclusive_sum32(int v, int* s_wave)
{
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int incl = static_cast<int>(wave_inclusive_sum32(static_cast<uint32_t>(v)));
  if (lane == 63) s_wave[wave] = incl;
  __syncthreads();
  int before = 0;
  for (int w = 0; w < kT / 64; w++) before += w < wave ? s_wave[w] : 0;
  return before + incl - v;
}

// The order of cand_better among equal gains as one number, for fewer than 2^26 bins: larger wins, none is 0.
__device__ __forceinline__ unsigned tie_key_of_bin(int bin)
{
  return (static_cast<unsigned>(bin & 511) << 17 | static_cast<unsigned>(0x1ffff - (bin >> 9))) + 1u;
}

__device__ __forceinline__ int bin_of_tie_key(unsigned key)
{
  return static_cast<int>(((key - 1u) >> 17) | ((0x1ffffu - ((key - 1u) & 0x1ffffu)) << 9));
}

// Split proposals of one feature by one workgroup (build_tree.cu:867-964): the sampled rows' values,
// sorted on order-preserving keys, without repetitions.
struct SampleSpec {
  int S;
  int32_t seed;
  int64_t dataset_rows, row_offset, n_rows;
  int F;
};
constexpr int kRankSortMax = 512;  // samples (a power of two that holds them) sorted by counting the smaller ones; more: a bitonic network
template <typename T>
constexpr int kProposalScratch = 2 * sizeof(T) + 4;  // bytes of LDS per sample (of P, the power of two)

// Returns their number; *proposals points to them in the LDS (the last one stands for +inf,
// build_tree.cu:953-956). P: power of two that holds S, at most 2 * kT. s_wave: kT / 64 ints. smem: aligned to 16 bytes
template <typename T, int kT>
__device__ __forceinline__ int feature_proposals(const T* __restrict__ X, const SampleSpec& a, int f, int P,
                                                 unsigned char* smem, int* s_wave, const T** proposals)
{
  using Key   = typename KeyOf<T>::type;
  Key* s_in   = reinterpret_cast<Key*>(smem);           // [P] as drawn; later the distinct values
  Key* s_key  = s_in + P;                               // [P] sorted
  int* s_rank = reinterpret_cast<int*>(s_key + P);      // [P]
  __shared__ int s_n;
  const int tid = threadIdx.x;
  const bool few = P >= 8 && P <= kRankSortMax && P <= kT;
  unsigned met   = 0;  // 1: a NaN, 2: a negative zero
  // the sampled rows (build_tree.cu:882-898)
  for (int i = tid; i < P; i += kT) {
    Key key = ~Key(0);
    if (i < a.S) {
      uint32_t x = minstd_seed(static_cast<uint32_t>(a.seed));
      x          = minstd_next(minstd_discard(x, static_cast<uint64_t>(i)));
      const double u    = uniform01(x);
      const double b    = static_cast<double>(a.dataset_rows - 1) + 1.0;
      const int64_t row = static_cast<int64_t>((u * (b - 0.0)) + 0.0) - a.row_offset;
      key               = to_key(row >= 0 && row < a.n_rows ? X[row * a.F + f] : T(0));
    }
    s_in[i] = key;
    if (few) {
      s_key[i]  = ~Key(0);
      s_rank[i] = 0;
      const T v = from_key(key);
      met |= i < a.S ? (v != v ? 1u : 0u) | (key == to_key(T(-0.0)) ? 2u : 0u) : 0u;
    } else {
      s_key[i] = key;
    }
  }
  const int wave = tid >> 6, lane = tid & 63;
  if (few) {
    const unsigned wave_met = (__any(met & 1u) ? 1u : 0u) | (__any(met & 2u) ? 2u : 0u);
    if (lane == 0) s_wave[wave] = static_cast<int>(wave_met);
  }
  __syncthreads();
  if (few) {
    met = 0;
    for (int w = 0; w < kT / 64; w++) met |= static_cast<unsigned>(s_wave[w]);
  }
  const bool by_count = few && (met & 1u) == 0;
  if (by_count) {
    // A value's place is the number of smaller samples, the same for equal ones, of which one is wanted: a comparison and an addition with its
    // carry each, which is what this takes, and places that stay empty. Several threads share the counting. (256 samples, 1024
    // threads: 4100 cycles; with the index of equal samples compared as well 10,100. Launches with 256 samples, 1000 x 10 f64 11.1 us and
    // 8.2, 100,000 x 32 14.2 and 10.7; with 512, 1008 x 151 24.1 and 13.8. Not with a NaN, which is not equal to itself. By lanes that
    // are read in turn, or searches among sorted runs of 64, 9100 and 12,100 cycles: a chain of instructions of one or few waves.)
    constexpr int kWide = 16 / sizeof(Key);
    struct alignas(16) Wide {
      Key v[kWide];
    };
    const int shift = 31 - __builtin_clz(P), parts = P >= 64 && kT > P ? min(kT >> shift, P / kWide) : 1, per = P / parts;
    if (tid < P * parts) {
      const int i          = tid & (P - 1);
      const Key mine       = s_in[i];
      const Wide* const from = reinterpret_cast<const Wide*>(s_in + (tid >> shift) * per);
      int before = 0;
#pragma unroll 4
      for (int w = 0; w < per / kWide; w++) {
        const Wide o = from[w];
#pragma unroll
        for (int u = 0; u < kWide; u++) before += o.v[u] < mine ? 1 : 0;
      }
      if (i < a.S) atomicAdd(&s_rank[i], before);
    }
    __syncthreads();
    if (tid < a.S) s_key[s_rank[tid]] = s_in[tid];
    __syncthreads();
  } else {
    if (few) {
      for (int i = tid; i < P; i += kT) s_key[i] = s_in[i];
      __syncthreads();
    }
    for (int size = 2; size <= P; size <<= 1)
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        for (int i = tid; i < P / 2; i += kT) {
          const int lo = 2 * i - (i & (stride - 1)), hi = lo + stride;
          const bool up = (lo & size) == 0;
          const Key x = s_key[lo], y = s_key[hi];
          if ((x > y) == up) {
            s_key[lo] = y;
            s_key[hi] = x;
          }
        }
        __syncthreads();
      }
  }
  T* s_prop = reinterpret_cast<T*>(s_in);
  if (by_count) {
    // those that are left lie apart, and zeros of either sign are equal
    const Key key   = tid < a.S ? s_key[tid] : ~Key(0);
    const bool keep = key != ~Key(0) && !(key == to_key(T(0.0)) && (met & 2u) != 0);
    const unsigned long long kept = __ballot(keep);
    if (lane == 0) s_wave[wave] = __popcll(kept);
    __syncthreads();
    int at = __popcll(kept & ((1ull << lane) - 1)), n = 0;
    for (int w = 0; w < kT / 64; w++) {
      at += w < wave ? s_wave[w] : 0;
      n += s_wave[w];
    }
    if (keep) s_prop[at] = from_key(key);
    __syncthreads();
    *proposals = s_prop;
    return n;
  }
  // drop values equal to their predecessor; two consecutive samples per thread
  T v[2] = {T(0), T(0)};
  bool keep[2];
  int mine = 0;
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int i = 2 * tid + u;
    keep[u]     = false;
    if (i < a.S) {
      v[u]    = from_key(s_key[i]);
      keep[u] = i == 0 || !(v[u] == from_key(s_key[i - 1]));
    }
    mine += keep[u] ? 1 : 0;
  }
  int at = block_exclusive_sum32<kT>(mine, s_wave);
  if (tid == kT - 1) s_n = at + mine;
#pragma unroll
  for (int u = 0; u < 2; u++)
    if (keep[u]) s_prop[at++] = v[u];
  __syncthreads();
  *proposals = s_prop;
  return s_n;
}

// A whole number as 64 bits: one conversion where it fits 32, as all but a value that ends the call does.
__device__ __forceinline__ int64_t whole_to_i64(double v)
{
  if (__builtin_expect(fabs(v) <= 2147483647.0, 1)) return static_cast<int32_t>(v);
  asm volatile("");  // (a branch: the general conversion is eight instructions)
  return static_cast<int64_t>(v);
}
// One stochastic rounding of a (grad, hess) pair (build_tree.cu:112-129).
__device__ __forceinline__ void quantise_pair(double grad, double hess, double sg, double sh, int64_t seed, int64_t row,
                                              int64_t k, int64_t* qg, int64_t* qh)
{
  uint32_t x = minstd_seed(static_cast<uint32_t>(static_cast<uint64_t>(gpair_seed(seed, row, k))));
  const double scaled_grad    = grad * sg;
  const double scaled_hess    = hess * sh;
  const double grad_remainder = scaled_grad - floor(scaled_grad);
  const double hess_remainder = scaled_hess - floor(scaled_hess);
  x   = minstd_next(x);
  *qg = whole_to_i64(floor(scaled_grad) + static_cast<double>(uniform01(x) < grad_remainder));
  x   = minstd_next(x);
  *qh = whole_to_i64(floor(scaled_hess) + static_cast<double>(uniform01(x) < hess_remainder));
}

// ---- bin search (see build_cells_kernel for the table)

// The cell of a value. Equal cells over the range of the proposals serve evenly spread columns only:
// with a long tail (lognormal columns) most proposals crowd into a few of them, the table's start then
// lies far before the bin and nearly every wave has a lane that walks on (4M x 100 lognormal values: 1.74 ms
// where uniform ones took 0.54). So the axis is bent first:
//   d = (x - centre) * scale,  g = sign(d) * log2(1 + |d|) in its piecewise linear form
// (the bits of the float 1 + |d| read as an integer), which is exactly linear for |d| <= 1 and
// logarithmic beyond; build_cells_kernel picks centre and scale per feature, a scale that keeps the
// whole range inside |d| <= 1 being one of its choices. The cell is then g * invw + nlo clamped to
// [0, cmax]. Every step is monotone non-decreasing in x (a fused multiply-add with a non-negative factor
// rounds once, and rounding, the bit pattern of positive floats and clamping keep order), and table
// construction and lookup share this function, which is all that exactness needs. NaN goes to cell 0.
template <typename T>
struct CellMap {
  T scale, shift;      // d = x * scale + shift
  float invw, nlo;     // t = g * invw + nlo
};
__device__ __forceinline__ float bend(float d)
{
  const int k = __float_as_int(fabsf(d) + 1.0f) - 0x3f800000;
  return copysignf(static_cast<float>(k), d);
}
template <typename T>
__device__ __forceinline__ float bend_axis(T x, T scale, T shift)
{
  // the median of (x, -max, max) clamps infinities; with a NaN operand it is the minimum of the others
  if constexpr (sizeof(T) == 4) {
    constexpr float kMax = std::numeric_limits<float>::max();
    return bend(fmaf(__builtin_amdgcn_fmed3f(x, -kMax, kMax), scale, shift));
  } else {
    constexpr double kMax = std::numeric_limits<double>::max();
    const double v        = x > -kMax ? x : -kMax;  // false for NaN
    return bend(static_cast<float>(fma(v, scale, shift)));
  }
}
template <typename T>
__device__ __forceinline__ int cell_of(T x, T scale, T shift, float invw, float nlo, float cmax)
{
  return static_cast<int>(__builtin_amdgcn_fmed3f(fmaf(bend_axis(x, scale, shift), invw, nlo), 0.0f, cmax));
}
// Without the bend, for features whose proposals spread evenly: six vector instructions less per value,
// which the binning pass feels (4M x 100 uniform values: 0.60 ms bent, 0.54 straight).
template <typename T>
__device__ __forceinline__ int straight_cell_of(T x, T a, T b, float cmax)
{
  return static_cast<int>(__builtin_amdgcn_fmed3f(static_cast<float>(fma(x, a, b)), 0.0f, cmax));
}

// A table holds, for every 32 cells, the number of proposals in all cells before them (y) and a bit per proposal of theirs (x), at
// its cell or, where another one has taken that, at the next free cell of the entry (at none behind the last). A value's start, y and
// the bits below its cell, so never exceeds the number of proposals below it, and where its cell's bit is not set it is that number.
// A field whose width the hardware takes modulo 32 and a count that adds give the start in two
// vector instructions (six with 16 cells and the count in one word).
constexpr int kCellsPerEntry = 32;
constexpr int kCellShift     = 5;  // log2(kCellsPerEntry); cells are never negative

__device__ __forceinline__ int table_start(const uint2& entry, int cell)
{
  return static_cast<int>(entry.y) + __popc(__builtin_amdgcn_ubfe(entry.x, 0, static_cast<unsigned>(cell)));
}
// all ones where the cell's bit is set, else zero: the value's bin then is the start itself
__device__ __forceinline__ int table_occupied(const uint2& entry, int cell)
{
  return __builtin_amdgcn_sbfe(static_cast<int>(entry.x), static_cast<unsigned>(cell), 1);
}

// The bent map of a feature is the one of a few candidates (linear; logarithmic on both sides of a
// centre at the low end, the median or the high end of the proposals, at three scales) that leaves the
// fewest proposals in a cell with their predecessor: the proposals are a sample of the column, so they
// say where its values fall.
constexpr int kCellMaps = 10;
template <typename T>
__device__ inline CellMap<T> cell_map_candidate(int c, const T* p, int n, float cells)
{
  CellMap<T> m{T(0), T(0), 0.0f, 0.0f};
  if (n < 3) return m;  // at least two finite proposals (the last one is +inf)
  const T lo = p[0], hi = p[n - 2], mid = p[(n - 1) / 2];
  const T width = hi - lo;
  // (a -inf proposal, or a range that overflows: everything in cell 0)
  if (!(width > T(0) && width < std::numeric_limits<T>::infinity())) return m;
  T centre = lo, scale = T(1) / width;
  if (c > 0) {
    const int where = (c - 1) % 3, fine = (c - 1) / 3;
    centre          = where == 0 ? mid : (where == 1 ? lo : hi);
    // half of the proposals lie inside one unit of d (fine = 0), a quarter, an eighth
    const int q  = max(1, (n - 1) >> (2 + fine));
    const int at = (n - 1) / 2;
    T reach      = where == 0 ? (p[min(n - 2, at + q)] - p[max(0, at - q)]) / T(2)
                              : (where == 1 ? p[min(n - 2, 2 * q)] - lo : hi - p[max(0, n - 2 - 2 * q)]);
    if (!(reach > width * T(1e-6))) reach = width * T(1e-6);
    scale = T(1) / reach;
  }
  const T shift = -centre * scale;
  if (!(scale < std::numeric_limits<T>::infinity()) || !(shift - shift == T(0))) return m;
  const float g_lo = bend_axis(lo, scale, shift), g_hi = bend_axis(hi, scale, shift);
  const float invw = cells / (g_hi - g_lo);
  if (!(g_hi > g_lo) || !(invw < std::numeric_limits<float>::infinity())) return m;
  m.scale = scale;
  m.shift = shift;
  m.invw  = invw;
  m.nlo   = -g_lo * invw;
  return m;
}

// Proposals that share their cell with their predecessor under candidate c, counted by one wave; *map: the candidate. (A cell per proposal, its
// predecessor's from the lane before, and counts of lanes; with both cells formed by every lane, the lanes' counts added up by permutes and the best
// candidate formed again, the prologue of 100,000 x 32 took 11.2 us, now 10.0, and build_cells_kernel of 1,000,000 x 50 with 512 samples 18.0, now 16.4.)
template <typename T>
__device__ __forceinline__ int crowded_proposals(int c, const T* p, int n, int C, int lane, CellMap<T>* map)
{
  const CellMap<T> m = cell_map_candidate(c, p, n, static_cast<float>(C));
  if (lane == 0) *map = m;
  const float cmax = static_cast<float>(C - 1);
  int crowded = 0, last = -1;  // cell of the proposal before these
  for (int first = 0; first < n - 1; first += 64) {
    const int i      = min(first + lane, n - 2);
    const int cell   = cell_of(p[i], m.scale, m.shift, m.invw, m.nlo, cmax);
    const int before = __builtin_amdgcn_update_dpp(last, cell, 0x138, 0xf, 0xf, false);  // from the lane before, lane 0: last
    crowded += __popcll(__ballot(first + lane < n - 1 && cell == before));
    last = __builtin_amdgcn_readlane(cell, 63);
  }
  return crowded;
}

// Table of a feature under the cell function `cell`, by the whole workgroup. The first proposal of an
// entry says how many are before it (the cells of ascending proposals ascend), then a thread per entry places its bits.
struct CellScratch {  // LDS
  uint16_t cell[LBT_MAX_SPLIT_SAMPLES];
  int count[kMaxCells / kCellsPerEntry + 1];
};
template <typename T, typename CellFn>
__device__ __forceinline__ void write_cell_entries(const T* p, int n, int entries, CellScratch& s, uint2* table, CellFn cell)
{
  constexpr uint16_t kNan = 0xffff;  // sampled NaNs (in front of the last proposal) have no cell
  static_assert(kMaxCells < kNan, "a cell fits the scratch");
  for (int i = threadIdx.x; i < n; i += blockDim.x) s.cell[i] = p[i] == p[i] ? static_cast<uint16_t>(cell(p[i])) : kNan;
  for (int e = threadIdx.x; e <= entries; e += blockDim.x) s.count[e] = n;
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    if (s.cell[i] == kNan) continue;
    int before = i - 1;
    while (before >= 0 && s.cell[before] == kNan) before--;
    const int last = s.cell[i] >> kCellShift;
    for (int e = before < 0 ? 0 : (s.cell[before] >> kCellShift) + 1; e <= last; e++) s.count[e] = i;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < entries; e += blockDim.x) {
    const int i0 = s.count[e], i1 = s.count[e + 1];
    uint32_t bits = 0;
    int at        = -1;
    for (int i = i0; i < i1; i++) {
      if (s.cell[i] == kNan) continue;
      at = max(static_cast<int>(s.cell[i]) & (kCellsPerEntry - 1), at + 1);
      if (at >= kCellsPerEntry) break;
      bits |= 1u << at;
    }
    table[e] = make_uint2(bits, static_cast<uint32_t>(i0));
  }
  __syncthreads();
}

// Number of proposals in [p, p+n) that are < x (branch-free, fixed trip count).
template <typename T>
__device__ inline int count_less(const T* p, int n, T x, int steps)
{
  int lo = 0;
  for (int s = 0; s < steps; s++) {
    int half = n >> 1;
    bool go  = n > 0 && p[lo + half] < x;
    lo       = go ? lo + half + 1 : lo;
    n        = go ? n - half - 1 : half;
  }
  return lo;
}


// The tiles of a batch, a workgroup of kPlanThreads for 256 of them: every workgroup
// repeats the count and the scan of the nodes' tiles (a few loads per thread) instead of waiting
// for a launch that does it once, then writes the descriptors of its own 256 tiles. Workgroup 0
// also leaves the batch's totals and clears the counters of the launch that follows.
// Bound by latency: the nodes' sums and segments, a scan, the descriptors. The scan is one barrier, the totals are summed by
// waves, what they are added to is asked for at the start, and up to 256 nodes a descriptor needs nothing more from memory
// (1,000,000 x 50, 8 to 256 nodes: 4.7, 5.7, 6.8, 10.5, 7, 9 us, now 4.8, 3.9, 3.6, 3.6, 3.3, 3.9).
__device__ __forceinline__ void plan_tiles_block(const PlanArgs& a, int block)
{
  const int j0 = a.j0, j1 = a.j1, level_first = a.level_first, tile_rows = a.tile_rows;
  const int32_t* __restrict__ const seg       = a.seg;
  const I64Pair* __restrict__ const node_sums = a.node_sums;
  const HistView& hist                        = a.hist;
  int32_t* const pair_sync                    = a.pair_sync;
  int32_t* const partial_count                = a.partial_count;
  int32_t* const partial_list_count           = a.partial_list_count;
  LevelMeta* const meta                       = a.meta;
  LevelMeta* const level_total                = a.level_total;
  int4* const tiles                           = a.tiles;
  __shared__ int s_scan[kPlanThreads];
  __shared__ int2 s_seg[kPlanThreads];
  __shared__ int s_wave[kPlanThreads / 64];
  __shared__ int64_t s_sums[3][kPlanThreads / 64];
  const bool first_wg = block == 0;
  LevelMeta level_before{};
  if (first_wg) {
    if (threadIdx.x == 0) level_before = *level_total;
    if (pair_sync != nullptr)
      for (int i = threadIdx.x; i < kPairSyncSlots; i += kPlanThreads) pair_sync[i] = 0;
    if (partial_count != nullptr) {
      if (threadIdx.x == 0) *partial_count = 0;
      for (int i = threadIdx.x; i < kPartialMaxLists; i += kPlanThreads) partial_list_count[i] = 0;
    }
  }
  const int n     = j1 - j0;
  const int per   = (n + kPlanThreads - 1) / kPlanThreads;
  const int begin = j0 + min(n, static_cast<int>(threadIdx.x) * per);
  const int end   = j0 + min(n, (static_cast<int>(threadIdx.x) + 1) * per);
  auto tiles_of = [&](int j, int& rows, bool& built) {
    rows  = seg[j + 1] - seg[j];
    built = hist.builds(level_first + j, node_sums);
    return built ? (rows + tile_rows - 1) / tile_rows : 0;
  };
  int mine = 0;
  int64_t rb = 0, rc = 0, nb = 0;
  for (int j = begin; j < end; j++) {
    int rows;
    bool built;
    mine += tiles_of(j, rows, built);
    rb += rows;
    if (built && rows > 0) {
      rc += rows;
      nb += 1;
    }
  }
  // (a thread's only node: its tiles are written from here, by whoever owns them)
  s_seg[threadIdx.x] = begin < end ? make_int2(seg[begin], seg[begin + 1]) : make_int2(0, 0);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int before = block_exclusive_sum32<kPlanThreads>(mine, s_wave);
  s_scan[threadIdx.x] = before + mine;
  if (first_wg) {
    rb = wave_inclusive_sum(rb);
    rc = wave_inclusive_sum(rc);
    nb = wave_inclusive_sum(nb);
    if (lane == 63) {
      s_sums[0][wave] = rb;
      s_sums[1][wave] = rc;
      s_sums[2][wave] = nb;
    }
  }
  __syncthreads();
  const int total = s_scan[kPlanThreads - 1];
  if (first_wg && threadIdx.x == 0) {
    int64_t sum[3] = {0, 0, 0};
    for (int q = 0; q < 3; q++)
      for (int w = 0; w < kPlanThreads / 64; w++) sum[q] += s_sums[q][w];
    meta->n_tiles         = total;
    meta->instances       = sum[0];
    meta->built_instances = sum[1];
    meta->built_nodes     = sum[2];
    level_total->instances       = level_before.instances + sum[0];
    level_total->built_instances = level_before.built_instances + sum[1];
    level_total->built_nodes     = level_before.built_nodes + sum[2];
  }
  const int tile = block * kPlanThreads + threadIdx.x;
  if (tile >= total) return;
  // the thread whose run of nodes holds the tile: the last one whose inclusive count exceeds it
  int lo = 0, hi = kPlanThreads - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (s_scan[mid] > tile)
      hi = mid;
    else
      lo = mid + 1;
  }
  if (per == 1) {
    const int2 sg = s_seg[lo];
    const int r0  = sg.x + (tile - (lo > 0 ? s_scan[lo - 1] : 0)) * tile_rows;
    tiles[tile]   = make_int4(level_first + j0 + lo, r0, min(sg.y, r0 + tile_rows), sg.y - sg.x);
    return;
  }
  int run       = lo > 0 ? s_scan[lo - 1] : 0;  // first tile of that thread's run
  const int b2  = j0 + min(n, lo * per);
  const int e2  = j0 + min(n, (lo + 1) * per);
  for (int j = b2; j < e2; j++) {
    int rows;
    bool built;
    const int t = tiles_of(j, rows, built);
    if (tile < run + t) {
      const int seg_lo = seg[j], seg_hi = seg[j + 1];
      const int r0     = seg_lo + (tile - run) * tile_rows;
      tiles[tile]      = make_int4(level_first + j, r0, min(seg_hi, r0 + tile_rows), seg_hi - seg_lo);
      return;
    }
    run += t;
  }
}

}  // namespace lbt
