// Histogram stage of BuildTreeTask: for every row of a node whose histogram is
// built, every feature f and output k,
//   hist[node][k][lower_bound(proposals of f, X[row][f])] += quantised (g, h)
// (rapidsai/legate-boost src/models/tree/build_tree.cu:213-577, build_tree.h:178-185).
//
// Layout of the work on gfx950:
//   * The lower bound of a value does not depend on the tree level, so it is
//     computed once: a root pass (bin_rows_kernel) reads X in whole rows and
//     stores the feature-relative bin of every value in one or two bytes (the
//     bin cache). The histograms of all levels, the root included, are then
//     accumulated from the cache (binned_histogram_kernel); a level reads a
//     quarter of the bytes X would cost and does no search.
//   * Bin search: a monotone function of the value, fitted to the feature's proposals, gives a
//     cell of a per-feature table that holds the number of proposals in cells before it; a
//     short forward probe over the proposals finishes the search. Any monotone cell function
//     is exact here; the table is built on the device with the same function. Proposals
//     and tables of a search group of features sit in LDS (all 100 features of a
//     10M x 100 matrix with 256 proposals each are one group).
//   * The packed sub-histogram of a histogram group of features (8 bytes per bin)
//     is the only LDS state of the histogram kernel. (grad, hess) of a row are
//     one 64-bit word (grad * 2^32 + hess, both signed; see pack_pair)
//     added with a single LDS atomic; the sub-histogram is merged into the int64
//     histogram with global atomics when the workgroup moves to another node.
//     Before either half could overflow
//     (rows * max |q| >= 2^31) it is merged early; rows of tiny nodes go
//     straight to global atomics.
//   * The cache is stored row by row, the records of a row's histogram groups side by side, in one plane per search group
//     where the histogram groups lie within the search groups (see hist_prepare).
//     A record holds the group's bins and, for single-output trees, the row's
//     packed (grad, hess), padded to 32 bytes: 64 bytes for 52 features. A
//     row gathered at a deep level then costs one cache line per group and the
//     gradient pair comes with it instead of through a second gather.
//   * A histogram workgroup owns (a contiguous range of row tiles) x (group) x
//     (output). All workgroups are resident at once. A lane is tied to 16 bytes
//     of the record and walks rows; a tile is one pass of the workgroup (a few
//     rows per lane); the loads of the next tile and the row indices of the one
//     after are issued before the current tile is processed.
#include "lbt_device.h"
#include "lbt_internal.h"

#include <algorithm>
#include <cstring>
#include <type_traits>

namespace lbt {
namespace {

constexpr int kSmallNodeRows = 64;  // below this a node goes straight to global atomics
constexpr int kUnroll        = 4;   // rows per lane and tile, search kernels
constexpr int kBinnedUnroll  = 8;   // rows per lane and tile, histogram kernel (halved for 16-byte loads)
constexpr int kLinearProbes  = 8;   // forward probes before falling back to a binary search
constexpr int kPairSyncTiles = 8;   // tiles between two meeting points of the root launch's workgroups
constexpr int kPairSyncSpins = 64;  // polls (about 0.9 us apart) a workgroup waits at one
constexpr int kProbePad      = 3;   // +inf entries behind every feature's proposals in the binning pass
constexpr int kProbeSlack    = 8;   // further entries behind the last feature that a probe window may touch

// For the nodes [j0, j1) of the current level (level-local indices): decides
// which are built (build_tree.h:92-104) and cuts their row segments into tiles
// of tile_rows rows. tile_start[j - j0] = first tile of node j;
// tile_start[j1 - j0] = total.
__global__ void __launch_bounds__(kPlanThreads)
  plan_tiles_kernel(int j0, int j1, int level_first, const int32_t* seg, const I64Pair* node_sums,
                    HistView hist, int tile_rows, int32_t* tile_start, LevelMeta* meta, LevelMeta* level_total)
{
  // every thread owns a run of consecutive nodes: it counts their tiles, the workgroup scans the
  // 256 counts once, and the thread walks its run again to write the starts
  __shared__ int s_scan[kPlanThreads];
  __shared__ unsigned long long s_rb, s_rc, s_nb;
  if (threadIdx.x == 0) s_rb = s_rc = s_nb = 0;
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
  unsigned long long rb = 0, rc = 0, nb = 0;
  for (int j = begin; j < end; j++) {
    int rows;
    bool built;
    mine += tiles_of(j, rows, built);
    rb += static_cast<unsigned long long>(rows);
    if (built && rows > 0) {
      rc += static_cast<unsigned long long>(rows);
      nb += 1;
    }
  }
  s_scan[threadIdx.x] = mine;
  __syncthreads();
  for (int off = 1; off < kPlanThreads; off <<= 1) {
    const int v = static_cast<int>(threadIdx.x) >= off ? s_scan[threadIdx.x - off] : 0;
    __syncthreads();
    s_scan[threadIdx.x] += v;
    __syncthreads();
  }
  int run = s_scan[threadIdx.x] - mine;
  for (int j = begin; j < end; j++) {
    int rows;
    bool built;
    tile_start[j - j0] = run;
    run += tiles_of(j, rows, built);
  }
  if (rb != 0) atomicAdd(&s_rb, rb);
  if (rc != 0) atomicAdd(&s_rc, rc);
  if (nb != 0) atomicAdd(&s_nb, nb);
  __syncthreads();
  if (threadIdx.x == 0) {
    const int total       = s_scan[kPlanThreads - 1];
    tile_start[j1 - j0]   = total;
    meta->n_tiles         = total;
    meta->instances       = s_rb;
    meta->built_instances = s_rc;
    meta->built_nodes     = s_nb;
    level_total->instances += s_rb;
    level_total->built_instances += s_rc;
    level_total->built_nodes += s_nb;
  }
}

// One descriptor per tile, so that the histogram kernels need no search while they walk:
// (node, first row, end row, rows of the node), indexed like the tiles.
__global__ void __launch_bounds__(kPlanThreads)
  expand_tiles_kernel(int j0, int n_nodes, int level_first, const int32_t* seg, const int32_t* tile_start,
                      const LevelMeta* meta, int tile_rows, int4* tiles, int32_t* pair_sync, int32_t* partial_count,
                      int32_t* partial_list_count)
{
  // the arrival counters of the launch that follows start from zero
  if (blockIdx.x == 0 && pair_sync != nullptr)
    for (int i = threadIdx.x; i < kPairSyncSlots; i += kPlanThreads) pair_sync[i] = 0;
  if (blockIdx.x == 0 && partial_count != nullptr) {
    if (threadIdx.x == 0) *partial_count = 0;
    for (int i = threadIdx.x; i < kPartialMaxLists; i += kPlanThreads) partial_list_count[i] = 0;
  }
  const int tile = blockIdx.x * kPlanThreads + threadIdx.x;
  if (tile >= meta->n_tiles) return;
  // last j with tile_start[j] <= tile
  int lo = 0, hi = n_nodes;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (tile_start[mid] <= tile)
      lo = mid;
    else
      hi = mid - 1;
  }
  const int j      = j0 + lo;
  const int seg_lo = seg[j], seg_hi = seg[j + 1];
  const int r0     = seg_lo + (tile - tile_start[lo]) * tile_rows;
  tiles[tile]      = make_int4(level_first + j, r0, min(seg_hi, r0 + tile_rows), seg_hi - seg_lo);
}

// Both of the above in one launch, for batches of up to kPlanFusedNodes nodes (plan_tiles_block)
constexpr int kPlanFusedNodes = 4096;
__global__ void __launch_bounds__(kPlanThreads) plan_expand_tiles_kernel(PlanArgs a) { plan_tiles_block(a, blockIdx.x); }

// Lookup table of a feature: the value range is cut into C fine cells (many more than there
// are proposals) and the table holds one entry per 32 cells (see table_start). For a value in cell c,
//   start = count(entry of c) + popcount(bits of the entry below c)
// never exceeds the number of proposals below the value (a proposal in an earlier cell is
// smaller than every value of a later cell, and counted at its cell or later),
// so the lower bound lies at or after start and is found by comparing the next few
// proposals; with 8 cells per proposal three comparisons almost always suffice.
// Small tables of the host that travel with a launch (a kernel's arguments may take 4 KB).
struct SmallTables {
  static constexpr int kMost = 4, kWords = 640;
  uint32_t* to[kMost];
  int at[kMost], words[kMost];
  int n, used;
  uint32_t data[kWords];
};

// One workgroup per feature.
// tables: [2][F][entries], the bent maps' tables first. A feature is straight when the plain linear map
// leaves few of its proposals in a cell with their predecessor (normal columns: one in seven); only
// then its second table is written, and a search group all of whose features are straight uses those.
// Maps: map_x [2][F][2] (bent: scale, shift; straight: a, b), map_t [F][2], straight [F].
// The next workgroup copies the host's small tables, which come with the launch, and finds the root's outputs; the others clear the
// first levels' histograms. Three launches and a copy from pinned memory, with 5 to 6 us of nothing on either side of that, were
// 41 us of a tree of 1,000,000 x 50, now 22 (a tree 1426 us, both together 1387; of 9001 x 50, depth 12, 663 and 625).
constexpr int kClearUnits = 4;  // 16-byte units of a thread that clears
template <typename T>
__global__ void __launch_bounds__(256)
  build_cells_kernel(const T* proposals, const int32_t* row_pointers, int F, int C, uint2* tables, T* map_x,
                     float* map_t, int32_t* straight, SmallTables small, RootArgs root)
{
  __shared__ T s_p[LBT_MAX_SPLIT_SAMPLES];
  __shared__ int s_crowded[kCellMaps];
  __shared__ CellMap<T> s_map[kCellMaps];
  __shared__ CellScratch s_cells;
  const int f = blockIdx.x;
  if (f == F) {
    for (int i = 0; i < small.n; i++)
      for (int w = threadIdx.x; w < small.words[i]; w += 256) small.to[i][w] = small.data[small.at[i] + w];
    if (root.leaf != nullptr) {
      if (threadIdx.x < 2)
        __hip_atomic_store(root.host_stats + threadIdx.x, root.qstats[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      for (int k = threadIdx.x; k < root.K; k += 256) {
        const double G = static_cast<double>(root.node_sums[k].grad) * root.scales[2];
        const double H = static_cast<double>(root.node_sums[k].hess) * root.scales[3];
        root.leaf[k]   = calculate_leaf_value(G, H, root.l1, root.l2);
      }
    }
    return;
  }
  if (f > F) {
    const int64_t first = static_cast<int64_t>(f - F - 1) * (256 * kClearUnits) + threadIdx.x;
#pragma unroll
    for (int u = 0; u < kClearUnits; u++)
      if (first + u * 256 < root.n16) root.clear[first + u * 256] = make_uint4(0, 0, 0, 0);
    return;
  }
  const int b0 = row_pointers[f];
  const int n  = row_pointers[f + 1] - b0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) s_p[i] = proposals[b0 + i];
  __syncthreads();
  const T* p       = s_p;
  const float cmax = static_cast<float>(C - 1);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int c = wave; c < kCellMaps; c += 4) {
    const int crowded = crowded_proposals(c, p, n, C, lane, &s_map[c]);
    if (lane == 0) s_crowded[c] = crowded;
  }
  __syncthreads();
  int best = 0;
  for (int c = 1; c < kCellMaps; c++)
    if (s_crowded[c] < s_crowded[best]) best = c;
  const CellMap<T> m = s_map[best];
  const int entries  = C / kCellsPerEntry;
  write_cell_entries(p, n, entries, s_cells, tables + static_cast<int64_t>(f) * entries,
                     [&](T x) { return cell_of(x, m.scale, m.shift, m.invw, m.nlo, cmax); });
  // candidate 0 stands for the straight map, whose cells differ from it by roundings only
  T a = T(0), b = T(0);
  bool even = 4 * s_crowded[0] <= n;
  if (n >= 3 && even) {
    const T lo = p[0], width = p[n - 2] - lo;
    if (width > T(0) && width < std::numeric_limits<T>::infinity()) a = static_cast<T>(C) / width;
    b = -lo * a;
    if (!(a < std::numeric_limits<T>::infinity()) || !(b - b == T(0))) a = b = T(0);
  }
  if (even)
    write_cell_entries(p, n, entries, s_cells, tables + static_cast<int64_t>(F + f) * entries,
                       [&](T x) { return straight_cell_of(x, a, b, cmax); });
  if (threadIdx.x == 0) {
    map_x[2 * f]           = m.scale;
    map_x[2 * f + 1]       = m.shift;
    map_x[2 * (F + f)]     = a;
    map_x[2 * (F + f) + 1] = b;
    map_t[2 * f]           = m.invw;
    map_t[2 * f + 1]       = m.nlo;
    straight[f]            = even ? 1 : 0;
  }
}

// What both kernels need to walk the tiles of a batch.
struct TileWalk {
  int j0;           // first level-local node of the batch
  int n_nodes;      // nodes in the batch
  int level_first;  // global index of level-local node 0
  int tile_rows;
  int rpp;       // rows per pass of a workgroup (tile_rows / rows per lane)
  int n_gk;      // groups * outputs
  int n_chunks;  // row-tile ranges
  bool all_resident;  // host side: the launch's workgroups all fit the chip at once
};

// Read-only inputs of the tile walk. They are separate __restrict__ kernel
// parameters (not struct members) so that the compiler can prove that no store of
// the kernel touches them and fetch the uniform ones through the scalar cache;
// vector loads here would force waits that also drain the prefetched row data.
#define LBT_WALK_PARAMS                                                                 \
  const int32_t* __restrict__ positions, const int4* __restrict__ tiles,                   \
    const LevelMeta* __restrict__ meta, const unsigned long long* __restrict__ qstats

struct Tile {
  int node;
  int r0, r1;
  int seg_rows;
};

// The workgroup keeps a window of tile descriptors in LDS and refills it when the walk
// runs past its end; reading a descriptor is then an LDS access, not a chain of dependent
// global loads that would stall every wave of the workgroup at the same time.
constexpr int kTileWindow = 256;

struct TileWindow {
  int4* s_tiles;
  const int4* tiles;
  int base;
  int t_end;
  __device__ void fill(int first)
  {
    base = first;
    __syncthreads();
    for (int i = threadIdx.x; i < kTileWindow && first + i < t_end; i += blockDim.x) s_tiles[i] = tiles[first + i];
    __syncthreads();
  }
  // all threads of the workgroup call this with the same, non-decreasing tile index
  __device__ Tile get(int tile)
  {
    if (tile - base >= kTileWindow) fill(tile);
    const int4 d = s_tiles[tile - base];
    Tile t;
    t.node     = d.x;
    t.r0       = d.y;
    t.r1       = d.z;
    t.seg_rows = d.w;
    return t;
  }
};

template <typename T>
struct HistArgs {
  TileWalk w;
  int F;
  int64_t n_rows;
  int K;
  const T* proposals;
  const int32_t* row_pointers;
  const int32_t* groups;  // feature groups: [n_groups+1]
  const uint2* tables;
  const T* map_x;      // scale, shift (see build_cells_kernel)
  const float* map_t;  // invw, nlo
  int cells;
  int search_steps;
  HistView hist;
};

template <typename T, int VEC>
struct VecOf;
template <>
struct VecOf<float, 4> {
  using type = float4;
};
template <>
struct VecOf<float, 2> {
  using type = float2;
};
template <>
struct VecOf<float, 1> {
  using type = float;
};
template <>
struct VecOf<double, 4> {
  using type = double4;
};
template <>
struct VecOf<double, 2> {
  using type = double2;
};
template <>
struct VecOf<double, 1> {
  using type = double;
};

// The same vectors for rows that start on a multiple of the element size only (a feature
// count that is no multiple of the vector width): loaded with element alignment.
template <typename T, int VEC>
struct __attribute__((packed, aligned(sizeof(T)))) LooseVec {
  T v[VEC];
};

// A (grad, hess) pair as one 64-bit addend: grad * 2^32 + hess, both signed. Sums of such
// words are sums of both halves as long as each total stays inside (-2^31, 2^31): the low
// 32 bits of the sum, read as a signed number, are the hess total, and what is left after
// taking it away is the grad total times 2^32. A negative hess (custom objectives) borrows
// from the high half when it is packed and gives the borrow back when it is unpacked.
__device__ __forceinline__ unsigned long long pack_pair(int grad, int hess)
{
  return (static_cast<unsigned long long>(static_cast<uint32_t>(grad + (hess >> 31))) << 32) |
         static_cast<unsigned long long>(static_cast<uint32_t>(hess));
}
__device__ __forceinline__ void unpack_pair(unsigned long long v, int32_t& grad, int32_t& hess)
{
  hess = static_cast<int32_t>(static_cast<uint32_t>(v));
  grad = static_cast<int32_t>(static_cast<uint32_t>(v >> 32)) - (hess >> 31);
}

// Merge of the packed LDS sub-histogram into the int64 histogram of a node.
__device__ inline void merge_sub_histogram(unsigned long long* s_hist, int nb, I64Pair* dst)
{
  // Workgroups that finish a node together would walk its bins in step and queue up on the
  // same cache lines: each one starts at a place of its own and wraps around.
  const int start = static_cast<int>((blockIdx.x * 2654435761u) % static_cast<unsigned>(nb));
  for (int t = threadIdx.x; t < nb; t += kHistThreads) {
    const int i          = t + start < nb ? t + start : t + start - nb;
    unsigned long long v = s_hist[i];
    if (v != 0) {
      int32_t gv, hv;
      unpack_pair(v, gv, hv);
      if (gv != 0) atomic_add_i64(&dst[i].grad, static_cast<int64_t>(gv));
      if (hv != 0) atomic_add_i64(&dst[i].hess, static_cast<int64_t>(hv));
      s_hist[i] = 0;
    }
  }
}

// The striped layout of the packed sub-histogram: word bin * W + p holds bin `bin` of the group's
// feature p, W a power of two (at least 16) that is not smaller than the group. The LDS serves a
// wave-level 64-bit atomic quarter wave by quarter wave, and the 16 lanes of a quarter conflict
// when two of them fall on the same pair of banks, i.e. when their word indices agree modulo 16.
// Here the index modulo 16 is the feature modulo 16, whatever the bin is, and a lane that holds
// 16 bins of a row takes them in an order of its own, byte (step + lane) mod 16 at every step:
// the 16 lanes of a quarter wave then always work on 16 different features modulo 16 and never
// conflict (7 cycles per wave-level atomic where data-dependent banks cost 10 to 11 and, with
// the same-address collisions of the 16 rows of a wave, 15 to 16 in the kernel).
//
// per > 0 (W = 64, groups of 33 to 64 features): the four lanes of a row take `per` features each, lane l the features from
// per * l on, instead of 16, 16, 16 and what is left (see spread_bins). The index modulo 16 then is 4 * (c modulo 4) + l for
// a lane's feature c < 12 (16 of 16), and the four rows of a quarter wave take c modulo 4 in four different orders. The one
// or two features of a lane beyond 12 have four or two copies in the last 16 of the 64 columns, the four rows of a
// quarter wave use different ones; whoever reads the array adds them (their sum has the range of a packed sum: it is the sum of the
// same rows). In the LDS columns 0..31 of all bins come first and columns 32..63 follow 64 KB behind: the address of a word is
// then a byte of the row's bins between two bytes that do not depend on them, one v_perm_b32.
struct Stripes {
  int log_w;  // log2 W; negative: the layout is [feature][bin], one run of bins per feature
  int bins;   // bins of the widest feature (rows of the striped array)
  int per;    // 0: column p is feature p; 12, 13, 14 or 16: features a lane takes
  __host__ __device__ int words() const { return bins << log_w; }
  // where the LDS has word i
  __device__ int place(int i) const { return per > 0 ? ((i & 32) << 8) + ((i >> 6) << 5) + (i & 31) : i; }
  // the feature of a column of a group of gs, -1: none, or a copy other than the first
  __device__ int feature(int col, int gs) const
  {
    int f = col;
    if (per > 0) {
      const int l = col & 3;
      if (col < 48 || per == 16)
        f = per * l + ((col >> 2) & 3) + 4 * (col >> 4);
      else if (per == 13)
        f = col < 52 ? 13 * l + 12 : gs;
      else if (per == 14)
        f = (col & 4) == 0 ? 14 * l + 12 + ((col - 48) >> 3) : gs;
      else
        f = gs;
    }
    return f < gs ? f : -1;
  }
  // per > 0, all threads of a workgroup: use(b, v) for bin b = wave, wave + 16, ... with v the sum in the thread's column (copies
  // added), columns without a feature among them; the array is cleared. A wave reads the 64 columns of a bin, each lane its own
  // word and the copies' from the other lanes: one lane that reads four words one after the other made the launches of 1,000,000 x 50
  // below the root 29 us long instead of 25.
  template <typename Use>
  __device__ void drain(unsigned long long* s_hist, Use use) const
  {
    constexpr int kWaves   = kHistThreads / 64;
    const bool copied      = (threadIdx.x & 63) >= 48;
    unsigned long long* at = s_hist + place(threadIdx.x);
    auto other = [](unsigned long long v, auto ctrl) {
      auto half = [](uint32_t w) { return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(w), decltype(ctrl)::value, 0xf, 0xf, true)); };
      return static_cast<unsigned long long>(half(static_cast<uint32_t>(v >> 32))) << 32 | half(static_cast<uint32_t>(v));
    };
    auto whole = [&](unsigned long long v) {
      unsigned long long sum = v;
      if (per == 13) {  // row_ror:8, row_ror:4: the four columns of a lane of the row
        sum += other(sum, std::integral_constant<int, 0x128>{});
        sum += other(sum, std::integral_constant<int, 0x124>{});
      } else if (per == 14) {  // row_ror:12: the column four further
        sum += other(sum, std::integral_constant<int, 0x12c>{});
      }
      return copied ? sum : v;
    };
    for (int b = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6); b < bins; b += kWaves, at += kWaves * 32) {
      const unsigned long long v = *at;
      *at = 0;
      use(b, whole(v));
    }
  }
};

// Merge of a striped sub-histogram into the int64 histogram of a node; s_off[p] is the place of
// feature p's first bin in the group's run of bins.
// sole_owner: no other workgroup adds to these bins and nothing has been added to them yet (the
// histogram starts from zero, parked parts of a node are added after the launch, and the caller
// does not claim ownership of a node of which it has already merged a part): the sums are stored
// as they are, which neither waits for a load nor occupies the L2's atomic units.
__device__ inline void merge_striped(unsigned long long* s_hist, const Stripes& st, const int* s_off, I64Pair* dst,
                                     bool sole_owner, int gs)
{
  auto put = [&](int at, unsigned long long v) {
    if (v == 0) return;
    int32_t gv, hv;
    unpack_pair(v, gv, hv);
    I64Pair* d = dst + at;
    if (sole_owner) {
      *d = I64Pair{gv, hv};
    } else {
      if (gv != 0) atomic_add_i64(&d->grad, static_cast<int64_t>(gv));
      if (hv != 0) atomic_add_i64(&d->hess, static_cast<int64_t>(hv));
    }
  };
  // columns past the group's features collect the adds of record padding
  if (st.per > 0) {
    const int f = st.feature(threadIdx.x & 63, gs), first = f >= 0 ? s_off[f] : 0;
    st.drain(s_hist, [&](int b, unsigned long long v) { if (f >= 0) put(first + b, v); });
    return;
  }
  const int words = st.words();
  for (int i = threadIdx.x; i < words; i += kHistThreads) {
    const int col              = i & ((1 << st.log_w) - 1);
    const unsigned long long v = s_hist[i];
    if (v != 0 && col < gs) {
      put(s_off[col] + (i >> st.log_w), v);
      s_hist[i] = 0;
    }
  }
}

// Where the workgroups of a launch park their sub-histograms for reduce_partials_kernel.
struct PartialSink {
  unsigned long long* partials;
  int32_t* lists;       // [list][kPartialListCap] slots of the list (node of the batch, group, output)
  int32_t* list_count;  // [list]
  int32_t* count;       // slots handed out
  int slots;            // 0: merge with atomics
  int stride;           // packed bins per slot
};

// Hands the packed sub-histogram over instead of adding it bin by bin: two 64-bit global
// atomics per bin and workgroup were a quarter of the histogram stage (the L2 completes about
// 5e10 of them per second). A workgroup takes a slot, copies its bins there as they are and
// clears them; a pass after the launch adds up the slots of every (node, group, output) with
// plain loads. Without a free slot the atomics do it. All threads of the workgroup call this.
__device__ inline void park_sub_histogram(unsigned long long* s_hist, int nb, I64Pair* dst, const PartialSink& sink,
                                          int tag, int* s_slot, bool sole_owner, const Stripes& st, const int* s_off,
                                          int gs)
{
  if (sole_owner && st.log_w >= 0) {
    merge_striped(s_hist, st, s_off, dst, true, gs);
    return;
  }
  if (sole_owner) {
    // every row of the node went through this workgroup in one piece: nobody else adds to these
    // bins, and nothing has been added to them yet, so the sums are stored as they are
    for (int i = threadIdx.x; i < nb; i += kHistThreads) {
      const unsigned long long v = s_hist[i];
      if (v != 0) {
        int32_t gv, hv;
        unpack_pair(v, gv, hv);
        dst[i]    = I64Pair{gv, hv};
        s_hist[i] = 0;
      }
    }
    return;
  }
  int slot = sink.slots;
  if (sink.slots > 0) {
    if (threadIdx.x == 0) {
      // a slot, and a place for it in the list of its (node, group, output)
      int got = atomicAdd(sink.count, 1);
      if (got < sink.slots) {
        const int at = atomicAdd(sink.list_count + tag, 1);
        if (at < kPartialListCap)
          sink.lists[static_cast<int64_t>(tag) * kPartialListCap + at] = got;
        else
          got = sink.slots;  // list full: this one goes the slow way
      }
      *s_slot = got;
    }
    __syncthreads();
    slot = *s_slot;
  }
  if (slot < sink.slots) {
    // the words as they lie in the LDS (striped: all of the array that is read again)
    const int words         = st.log_w >= 0 ? st.words() : nb;
    unsigned long long* out = sink.partials + static_cast<int64_t>(slot) * sink.stride;
    if (st.per > 0) {
      const int col   = threadIdx.x & 63;
      const bool wanted = st.feature(col, gs) >= 0;
      st.drain(s_hist, [&](int b, unsigned long long v) { if (wanted) out[b * 64 + col] = v; });
      return;
    }
    for (int i = threadIdx.x; i < words; i += kHistThreads) {
      out[i]    = s_hist[i];
      s_hist[i] = 0;
    }
  } else if (st.log_w >= 0) {
    merge_striped(s_hist, st, s_off, dst, false, gs);
  } else {
    merge_sub_histogram(s_hist, nb, dst);
  }
}

// Adds up the parked sub-histograms. Workgroup (x, y, z): bins x * 1024 .. of the list y =
// (node of the batch, group, output), every gridDim.z-th slot of the list starting with the
// z-th. With one workgroup per bin range (gridDim.z == 1) the totals are added plainly, no
// other workgroup touches those bins; a long list split over several workgroups (few lists:
// the levels near the root) adds them with atomics. Integer sums: any order gives the same.
__global__ void __launch_bounds__(kHistThreads)
  reduce_partials_kernel(PartialSink sink, int K, int n_groups, const int32_t* __restrict__ groups,
                         const int32_t* __restrict__ row_pointers, HistView hist, int first_node, Stripes st)
{
  const int tag = blockIdx.y;
  const int m   = min(sink.list_count[tag], kPartialListCap);
  if (static_cast<int>(blockIdx.z) >= m) return;
  const int n_gk  = n_groups * K;
  const int node  = first_node + tag / n_gk;
  const int gk    = tag - tag / n_gk * n_gk;
  const int group = gk / K, k = gk - gk / K * K;
  int bin0        = row_pointers[groups[group]];
  const int nb    = row_pointers[groups[group + 1]] - bin0;
  // `bin` is the word of the parked image; out_bin its place in the group's run of bins
  const int bin   = blockIdx.x * kHistThreads + threadIdx.x;
  int out_bin     = bin;
  if (st.log_w >= 0) {
    if (bin >= st.words()) return;
    const int p = st.feature(bin & ((1 << st.log_w) - 1), groups[group + 1] - groups[group]);
    const int f = groups[group] + p;
    const int b = bin >> st.log_w;
    if (p < 0 || b >= row_pointers[f + 1] - row_pointers[f]) return;
    out_bin = row_pointers[f] - bin0 + b;
  } else if (bin >= nb) {
    return;
  }
  const int32_t* __restrict__ list = sink.lists + static_cast<int64_t>(tag) * kPartialListCap;
  const unsigned long long* src    = sink.partials + bin;
  const int step                   = gridDim.z;
  int64_t g = 0, h = 0;
  int i = blockIdx.z;
  // eight slots at a time, so that their loads are in flight together
  for (; i + 7 * step < m; i += 8 * step) {
    unsigned long long v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = src[static_cast<int64_t>(list[i + u * step]) * sink.stride];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      int32_t gv, hv;
      unpack_pair(v[u], gv, hv);
      g += gv;
      h += hv;
    }
  }
  for (; i < m; i += step) {
    int32_t gv, hv;
    unpack_pair(src[static_cast<int64_t>(list[i]) * sink.stride], gv, hv);
    g += gv;
    h += hv;
  }
  I64Pair* dst = hist.at(node, k, bin0 + out_bin);
  if (step == 1) {
    dst->grad += g;
    dst->hess += h;
  } else {
    if (g != 0) atomic_add_i64(&dst->grad, g);
    if (h != 0) atomic_add_i64(&dst->hess, h);
  }
}

template <typename T, int VEC, bool kIdentityRows>
__global__ void __launch_bounds__(kHistThreads)
  histogram_kernel(HistArgs<T> a, LBT_WALK_PARAMS, const T* __restrict__ X, const int2* __restrict__ qgh)
{
  using Vec = typename VecOf<T, VEC>::type;
  extern __shared__ __align__(16) unsigned char smem_raw[];  // 16-byte aligned whatever static LDS precedes it
  const TileWalk& w = a.w;

  // workgroup -> (row-tile range, group, output). Linear workgroup ids are dealt
  // round-robin to the 8 XCDs, so id % 8 is the XCD; within an XCD consecutive
  // slots enumerate (group, output) of one row-tile range.
  const int xcd   = blockIdx.x & 7;
  const int slot  = blockIdx.x >> 3;
  const int gk    = slot % w.n_gk;
  const int chunk = (slot / w.n_gk) * 8 + xcd;
  const int group = gk / a.K;
  const int k     = gk % a.K;

  const int f0 = a.groups[group], f1 = a.groups[group + 1];
  const int gs   = f1 - f0;
  const int bin0 = a.row_pointers[f0];
  const int nb   = a.row_pointers[f1] - bin0;
  const int C    = a.cells;

  unsigned long long* s_hist = reinterpret_cast<unsigned long long*>(smem_raw);
  T* s_prop                  = reinterpret_cast<T*>(smem_raw + static_cast<size_t>(nb) * 8);
  uint2* s_cell              = reinterpret_cast<uint2*>(smem_raw + ((static_cast<size_t>(nb) * (8 + sizeof(T)) + 7) & ~size_t(7)));

  for (int i = threadIdx.x; i < nb; i += kHistThreads) {
    s_prop[i] = a.proposals[bin0 + i];
    s_hist[i] = 0;
  }
  {
    // tables of the group's features are contiguous
    const uint2* src  = a.tables + static_cast<int64_t>(f0) * (C / kCellsPerEntry);
    const int entries = gs * (C / kCellsPerEntry);
    for (int i = threadIdx.x; i < entries; i += kHistThreads) s_cell[i] = src[i];
  }

  const int lanes_per_row = (gs + VEC - 1) / VEC;
  const int lr            = threadIdx.x % lanes_per_row;
  const int rsub          = threadIdx.x / lanes_per_row;
  const bool active       = rsub < w.rpp;
  const int fl            = lr * VEC;  // first group-local feature of this lane

  T c_scale[VEC], c_shift[VEC];
  float c_invw[VEC], c_nlo[VEC];
  int c_cell[VEC], c_prop[VEC], c_end[VEC];
#pragma unroll
  for (int v = 0; v < VEC; v++) {
    int f     = min(f0 + fl + v, f1 - 1);
    c_scale[v] = a.map_x[2 * f];
    c_shift[v] = a.map_x[2 * f + 1];
    c_invw[v]  = a.map_t[2 * f];
    c_nlo[v]   = a.map_t[2 * f + 1];
    c_cell[v] = (f - f0) * (C / kCellsPerEntry);
    c_prop[v] = a.row_pointers[f] - bin0;
    c_end[v]  = a.row_pointers[f + 1] - bin0;
  }
  const float cmax = static_cast<float>(C - 1);
  const unsigned long long max_abs = qstats[0];

  const int n_tiles = meta->n_tiles;
  const int t_begin = static_cast<int>(static_cast<int64_t>(n_tiles) * chunk / w.n_chunks);
  const int t_end   = static_cast<int>(static_cast<int64_t>(n_tiles) * (chunk + 1) / w.n_chunks);

  int cur_node           = -1;
  unsigned long long acc = 0;  // rows added to the LDS copy since it was last merged
  __syncthreads();

  // Loads are unconditional (an index past the tile is clamped to the tile's first row and
  // the row is marked -1 afterwards), so that they issue back to back without branches.
  // The loaded index is not looked at until the data loads of the following iteration, so
  // nothing waits on it here; which rows of the tile exist is kept apart as a bit mask.
  auto load_rows = [&](const Tile& t, int (&row)[kUnroll]) -> unsigned {
    unsigned valid = 0;
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
      const int rr  = t.r0 + rsub + u * w.rpp;
      const bool ok = active && rr < t.r1;
      // at the root the order is still the identity: sorted index == row
      if constexpr (kIdentityRows)
        row[u] = ok ? rr : t.r0;
      else
        row[u] = positions[ok ? rr : t.r0];
      valid |= ok ? (1u << u) : 0u;
    }
    return valid;
  };
  auto load_data = [&](const int (&row)[kUnroll], Vec (&xv)[kUnroll], int2 (&q)[kUnroll]) {
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
      const int64_t rw = row[u];
      const T* xp      = X + rw * a.F + (f0 + fl);
      if constexpr (VEC == 1)
        xv[u] = *xp;
      else
        xv[u] = *reinterpret_cast<const Vec*>(xp);
      q[u] = qgh[rw * a.K + k];
    }
  };

  __shared__ int4 s_tile_window[kTileWindow];
  TileWindow win{s_tile_window, tiles, 0, t_end};
  win.fill(t_begin);
  Tile tc{}, tn{}, tnn{};
  int row_c[kUnroll], row_n[kUnroll], row_nn[kUnroll];
  Vec x_c[kUnroll], x_n[kUnroll];
  int2 q_c[kUnroll], q_n[kUnroll];
  unsigned valid_c = 0, valid_n = 0, valid_nn = 0;
#pragma unroll
  for (int u = 0; u < kUnroll; u++) row_c[u] = row_n[u] = row_nn[u] = 0;
  if (t_begin < t_end) {
    tc      = win.get(t_begin);
    valid_c = load_rows(tc, row_c);
    load_data(row_c, x_c, q_c);
  }
  if (t_begin + 1 < t_end) {
    tn      = win.get(t_begin + 1);
    valid_n = load_rows(tn, row_n);
  }

  for (int tile = t_begin; tile < t_end; tile++) {
    // issue the loads of the next tile and the row indices of the one after
    if (tile + 1 < t_end) load_data(row_n, x_n, q_n);
    if (tile + 2 < t_end) {
      tnn      = win.get(tile + 2);
      valid_nn = load_rows(tnn, row_nn);
    }

    const int nrows   = tc.r1 - tc.r0;
    const bool direct = tc.seg_rows < kSmallNodeRows ||
                        static_cast<unsigned long long>(nrows) * max_abs > 2147483647ULL;
    if (!direct) {
      if (tc.node != cur_node || (acc + nrows) * max_abs > 2147483647ULL) {
        __syncthreads();
        if (cur_node >= 0) merge_sub_histogram(s_hist, nb, a.hist.at(cur_node, k, bin0));
        __syncthreads();
        cur_node = tc.node;
        acc      = 0;
      }
      acc += nrows;
    }
    I64Pair* gdst = a.hist.at(tc.node, k, bin0);
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
      if (valid_c & (1u << u)) {
        const unsigned long long packed = pack_pair(q_c[u].x, q_c[u].y);
        T xs[VEC];
        if constexpr (VEC == 1) {
          xs[0] = x_c[u];
        } else if constexpr (VEC == 2) {
          xs[0] = x_c[u].x;
          xs[1] = x_c[u].y;
        } else {
          xs[0] = x_c[u].x;
          xs[1] = x_c[u].y;
          xs[2] = x_c[u].z;
          xs[3] = x_c[u].w;
        }
        int bin[VEC];
#pragma unroll
        for (int v = 0; v < VEC; v++) {
          const T x = xs[v];
          const int cell = cell_of(x, c_scale[v], c_shift[v], c_invw[v], c_nlo[v], cmax);
          int bn         = c_prop[v] + table_start(s_cell[c_cell[v] + (static_cast<unsigned>(cell) >> kCellShift)], cell);
          bool lt    = s_prop[bn] < x;
          int probes = 0;
          while (__any(lt)) {
            bn += lt ? 1 : 0;
            if (++probes == kLinearProbes) {
              bn += count_less(s_prop + bn, c_end[v] - bn, x, a.search_steps);
              break;
            }
            lt = s_prop[bn] < x;
          }
          bin[v] = bn;
        }
#pragma unroll
        for (int v = 0; v < VEC; v++) {
          if (direct) {
            atomic_add_i64(&gdst[bin[v]].grad, static_cast<int64_t>(q_c[u].x));
            atomic_add_i64(&gdst[bin[v]].hess, static_cast<int64_t>(q_c[u].y));
          } else {
            atomicAdd(&s_hist[bin[v]], packed);
          }
        }
      }
    }
    // rotate the pipeline
    tc      = tn;
    tn      = tnn;
    valid_c = valid_n;
    valid_n = valid_nn;
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
      row_c[u] = row_n[u];
      row_n[u] = row_nn[u];
      x_c[u]   = x_n[u];
      q_c[u]   = q_n[u];
    }
  }
  __syncthreads();
  if (cur_node >= 0) merge_sub_histogram(s_hist, nb, a.hist.at(cur_node, k, bin0));
}

// Root pass when the bin cache is in use: bins every value of X once and stores
// the feature-relative bins in the cache records. No histogram is kept here, so
// the LDS holds only proposals and lookup tables and a workgroup can cover all
// features of a row (100 features with 256 proposals each: one search group): X
// is then read in whole, contiguous rows. A lane bins VEC consecutive features,
// which always belong to one histogram group; further lanes have the zeros and, for
// single-output trees, the row's packed (grad, hess) that fill a record (see bin_lanes). The root histogram itself
// is accumulated from the cache like every other level.
//
// What bounds it: the memory, nearly. 10,000,000 x 100 f32 (4 GB read, 1.36 GB written) takes 1.21 ms, its loads and stores without any
// search 1.12, the same pattern of accesses in a stand-alone kernel 1.02 (1.43 before records were written by words of whole lines and
// the searches of a lane's values went side by side); 2,000,000 x 200 0.48 ms (0.74), 1,000,000 x 50 in two-byte bins 0.086 (0.114).
// what a lane of the quad has, for each of them two bits of kPerm
template <int kPerm>
__device__ __forceinline__ uint32_t quad_lane(uint32_t v)
{
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), kPerm, 0xf, 0xf, true));
}

template <typename T>
struct BinRowsArgs {
  int F;
  int64_t n_rows;
  const T* proposals;
  const int32_t* row_pointers;
  const int32_t* bin_feature;  // [bins] feature of every proposal
  const int32_t* sgroups;      // search groups: [n_sgroups+1]
  const uint2* tables;
  const T* map_x;      // maps and tables as build_cells_kernel writes them
  const float* map_t;
  const int32_t* straight;  // [F] the feature has a table for the straight cell function too
  int cells;
  int search_steps;
  int n_sgroups;
  int n_chunks;
  int rpp;                    // rows per pass of a workgroup
  int share;                  // lanes that share a record (kShared)
  const int2* lanes;          // lanes of a row of every search group (see bin_lanes)
  const RecInfo* rec;         // [histogram groups]
};

// kRagged: the feature count is no multiple of VEC. The last lane of a row then owns fewer
// than VEC features: it loads the VEC values that end with the row's last one and takes its
// own from their end, and its surplus bins are zeros in the record's padding. Rows then start
// on element boundaries only, so all lanes load with element alignment.
// kShared: rows of few features, whose records of 32 bytes their lanes share evenly (share_of_record).
template <typename T, int VEC, typename BinT, bool kRagged, bool kShared>
__global__ void __launch_bounds__(kHistThreads)
  bin_rows_kernel(BinRowsArgs<T> a, const T* __restrict__ X, const int2* __restrict__ qgh,
                  BinT* __restrict__ binned)
{
  using Vec = typename VecOf<T, VEC>::type;
  constexpr int kBatch = kUnroll * VEC <= 8 / (sizeof(T) / 4) ? kUnroll : 8 / (static_cast<int>(sizeof(T)) / 4) / VEC;  // rows searched side by side
  constexpr int kAhead = sizeof(T) * VEC == 32 ? 2 : kUnroll;  // rows whose values are on their way
  extern __shared__ __align__(16) unsigned char smem_raw[];  // 16-byte aligned whatever static LDS precedes it
  const int xcd   = blockIdx.x & 7;
  const int slot  = blockIdx.x >> 3;
  const int group = slot % a.n_sgroups;
  const int chunk = (slot / a.n_sgroups) * 8 + xcd;
  const int f0 = a.sgroups[group], f1 = a.sgroups[group + 1];
  const int gs   = f1 - f0;
  const int bin0 = a.row_pointers[f0];
  const int nb   = a.row_pointers[f1] - bin0;
  const int C    = a.cells;
  // LDS copy of the group's proposals: kProbePad entries of +inf in front of the first feature and behind every one, so that
  // a window of probes that starts anywhere in a feature stays ascending, and one at the front compares nothing
  T* s_prop        = reinterpret_cast<T*>(smem_raw);
  const int cell_at = ((nb + kProbePad * (gs + 1) + kProbeSlack) * static_cast<int>(sizeof(T)) + 7) & ~7;
  uint2* s_cell    = reinterpret_cast<uint2*>(smem_raw + cell_at);
  struct Proposal {
    T value;
    int feature;
  };
  copy_ahead<kHistThreads, 8>(
    nb, [&](int i) { return Proposal{a.proposals[bin0 + i], a.bin_feature[bin0 + i]}; },
    [&](int i, const Proposal& p) { s_prop[i + kProbePad * (p.feature - f0 + 1)] = p.value; });
  for (int i = threadIdx.x; i < kProbePad * (gs + 1) + kProbeSlack; i += kHistThreads) {
    const int f = min(i / kProbePad, gs);  // the pad in front of feature f; the slack follows the last one
    s_prop[a.row_pointers[f0 + f] - bin0 + i] = std::numeric_limits<T>::infinity();
  }
  // the straight cell function and its tables when every feature of the group has them
  bool bent_feature = false;
  for (int i = threadIdx.x; i < gs; i += kHistThreads) bent_feature |= a.straight[f0 + i] == 0;
  const bool bent = __syncthreads_or(bent_feature);
  {
    const uint2* src  = a.tables + static_cast<int64_t>(bent ? f0 : a.F + f0) * (C / kCellsPerEntry);
    const int entries = gs * (C / kCellsPerEntry);
    copy_ahead<kHistThreads, 8>(entries, [&](int i) { return src[i]; }, [&](int i, const uint2& e) { s_cell[i] = e; });
  }
  // The lanes of a row (see bin_lanes). Every lane that owns bins owns VEC real features (the last one of a ragged row: `mine` of them).
  const int2 head   = a.lanes[2 * group], plane = a.lanes[2 * group + 1];
  const int rsub    = threadIdx.x / head.y;
  const bool active = rsub < a.rpp;
  const int nth     = threadIdx.x % head.y;
  const int2 lane   = a.lanes[head.x + nth];
  constexpr int kOwn = VEC * static_cast<int>(sizeof(BinT));  // bytes of a lane's bins
  const int fb      = kShared || kOwn >= 4 ? lane.x : f0 + nth * VEC;  // first feature of this lane
  const int kind    = lane.y & 3;
  const int mine    = kRagged ? min(VEC, f1 - fb) : VEC;
  const int shift   = VEC - mine;     // its values are the last `mine` of the VEC it loads
  T c_scale[VEC], c_shift[VEC];
  float c_invw[VEC], c_nlo[VEC];
  int c_cell[VEC], c_prop[VEC];  // bytes from the start of the LDS to the feature's table and proposals
#pragma unroll
  for (int v = 0; v < VEC; v++) {
    const int f = kRagged ? min(fb + v, f1 - 1) : fb + v;
    const int at = 2 * (bent ? f : a.F + f);
    c_scale[v] = a.map_x[at];
    c_shift[v] = a.map_x[at + 1];
    c_invw[v]  = a.map_t[2 * f];
    c_nlo[v]   = a.map_t[2 * f + 1];
    c_cell[v] = cell_at + (f - f0) * (C / kCellsPerEntry) * static_cast<int>(sizeof(uint2));
    c_prop[v] = (a.row_pointers[f] - bin0 + kProbePad * (f - f0 + 1)) * static_cast<int>(sizeof(T));
  }
  const float cmax     = static_cast<float>(C - 1);
  // What a lane writes of a row are kWords words: its bins, zeros, or the row's gradient pair. A wave's stores so are one run of bytes
  // and nearly always whole cache lines, which is what the memory wants: with lanes for the bins alone and masked stores
  // of 16 bytes for what follows them 10,000,000 x 100 f32 took 1.32 ms, with the same pieces written by other waves 2.44 (lines
  // that reach the memory in parts), although a fifth fewer lanes search. kShared: its even share of the record's 32 bytes, of which the first 16 are
  // the bins of all its lanes. Bins of fewer than four bytes a lane are written byte by byte otherwise, their last lane filling the record (rows that
  // do not begin on a multiple of their values' size).
  constexpr int kWords   = kOwn >= 4 ? kOwn / 4 : 1;
  constexpr bool kByByte = !kShared && kOwn < 4;
  const int to_off       = lane.y >> 2;  // its bytes, from the row's first
  const bool pairs       = kShared && a.rec[0].q_off >= 0;
  // kByByte: the record's bytes behind the own bins up to the pair, and whether that follows
  int t_zero = 0, t_pair = -1;
  if (kByByte && kind == 1) {
    const RecInfo ri = a.rec[lane.x];
    t_zero = ri.in_row + ri.zero_end - to_off;
    t_pair = ri.q_off >= 0 ? ri.in_row + ri.q_off - to_off : -1;
  }
  // chunks start on multiples of 32 rows: with X itself aligned, the kilobyte a wave loads
  // then begins on a cache line whatever the row length is
  const int64_t r_begin = (a.n_rows * chunk / a.n_chunks) & ~int64_t(31);
  const int64_t r_end   = chunk + 1 == a.n_chunks ? a.n_rows : (a.n_rows * (chunk + 1) / a.n_chunks) & ~int64_t(31);
  // Inside the chunk rows are numbered from 0 and addressed by 32-bit byte offsets (the host
  // keeps a chunk's rows times the widest row below 2^31 bytes) from bases that are the same for the whole
  // workgroup; they advance by a uniform step from pass to pass instead of being multiplied out per row.
  const int n_local                  = static_cast<int>(r_end - r_begin);
  const unsigned char* const x_chunk = reinterpret_cast<const unsigned char*>(X + r_begin * a.F);
  // (trees of several outputs have no pair lanes, the words at the front of a row's pairs are read all the same)
  const unsigned char* const q_chunk = reinterpret_cast<const unsigned char*>(qgh + r_begin);
  const uint32_t row_bytes = static_cast<uint32_t>(a.F) * sizeof(T);
  const uint32_t rec_bytes = static_cast<uint32_t>(plane.x);
  // the search group's plane of the cache (or all of it)
  unsigned char* const b_chunk = reinterpret_cast<unsigned char*>(binned) + static_cast<int64_t>(plane.y) * kPlaneAlign + r_begin * rec_bytes;
  const uint32_t x_step    = static_cast<uint32_t>(a.rpp) * row_bytes;  // from one row of a pass to the next
  const uint32_t b_step    = static_cast<uint32_t>(a.rpp) * rec_bytes;
  const uint32_t x_lane    = static_cast<uint32_t>(fb - shift) * sizeof(T);
  const uint32_t x_last    = (n_local > 0 ? static_cast<uint32_t>(n_local - 1) * row_bytes : 0u) + x_lane;
  const int pass_rows      = a.rpp * kUnroll;
  __syncthreads();
  if (!active) return;

  // Pass p covers local rows (p * kUnroll + u) * rpp + rsub. A row's values are requested as soon as the row kAhead steps
  // before it has been searched, into the same registers. Rows past the chunk's end read its last row instead.
  uint32_t x_off = static_cast<uint32_t>(rsub) * row_bytes + x_lane;
  uint32_t q_off = static_cast<uint32_t>(rsub) * 8u + (kind == 3 ? 4u : 0u);
  const uint32_t q_step = static_cast<uint32_t>(a.rpp) * 8u;
  const uint32_t q_last = (n_local > 0 ? static_cast<uint32_t>(n_local - 1) * 8u : 0u) + (kind == 3 ? 4u : 0u);
  uint32_t b_off = static_cast<uint32_t>(rsub) * rec_bytes + static_cast<uint32_t>(to_off);
  auto load_row = [&](uint32_t at) {
    const uint32_t off = min(at, x_last);
    Vec xv;
    if constexpr (VEC == 1) {
      xv = *reinterpret_cast<const T*>(x_chunk + off);
    } else if constexpr (kRagged) {
      const LooseVec<T, VEC> lv = *reinterpret_cast<const LooseVec<T, VEC>*>(x_chunk + off);
      if constexpr (VEC == 2)
        xv = Vec{lv.v[0], lv.v[1]};
      else
        xv = Vec{lv.v[0], lv.v[1], lv.v[2], lv.v[3]};
    } else {
      xv = *reinterpret_cast<const Vec*>(x_chunk + off);
    }
    return xv;
  };
  auto take_values = [&](const Vec& from, T (&xs)[VEC]) {
    if constexpr (VEC == 1) {
      xs[0] = from;
    } else if constexpr (VEC == 2) {
      xs[0] = from.x;
      xs[1] = from.y;
    } else {
      xs[0] = from.x;
      xs[1] = from.y;
      xs[2] = from.z;
      xs[3] = from.w;
    }
    if constexpr (kRagged && VEC > 1) {
      // the lane with fewer features took the values that end with the row's last one
      T t[VEC];
#pragma unroll
      for (int v = 0; v < VEC; v++) t[v] = xs[v];
#pragma unroll
      for (int v = 0; v < VEC; v++) {
        T x = t[v];
#pragma unroll
        for (int sh = 1; sh < VEC; sh++)
          if (v + sh < VEC) x = shift == sh ? t[v + sh] : x;
        xs[v] = x;
      }
    }
  };
  const uint32_t pair_mask = kind >= 2 ? ~0u : 0u;
  // what a lane reads of a row's gradient pair, like its values: one word, or both
  using Pair = std::conditional_t<kWords == 2 || kOwn < 4 || kShared, int2, int>;
  auto load_pair = [&](uint32_t at) {
    if (kShared && !pairs) return Pair{};
    return *reinterpret_cast<const Pair*>(q_chunk + min(at, q_last));
  };
  // Loads come before the stores of a pass, in fixed numbers: a wait for loads behind stores would wait for these too.
  auto search_pass = [&](auto bent_cells, int first, Vec (&x_c)[kAhead], Pair (&q_c)[kAhead]) {
    uint32_t own[kUnroll][kWords];
    Pair pair_of[kShared ? kUnroll : 1];
    // The rows of a batch go through the search side by side, stage by stage: all reads of the tables, then all
    // probes. hipcc by itself takes one value after the other, two round trips through the LDS each.
#pragma unroll
    for (int u0 = 0; u0 < kUnroll; u0 += kBatch) {
      T xs[kBatch][VEC];
      int bn[kBatch][VEC], at[kBatch][VEC];
      {
        uint2 entry[kBatch][VEC];
        int cell[kBatch][VEC];
#pragma unroll
        for (int w = 0; w < kBatch; w++) {
          take_values(x_c[(u0 + w) % kAhead], xs[w]);
#pragma unroll
          for (int v = 0; v < VEC; v++) {
            const T x  = xs[w][v];
            cell[w][v] = decltype(bent_cells)::value ? cell_of(x, c_scale[v], c_shift[v], c_invw[v], c_nlo[v], cmax)
                                                     : straight_cell_of(x, c_scale[v], c_shift[v], cmax);
            // (the field as an instruction of its own: else its shift and the one of the entry's size become three)
            entry[w][v] = *reinterpret_cast<const uint2*>(
              smem_raw + (c_cell[v] + static_cast<int>(__builtin_amdgcn_ubfe(static_cast<unsigned>(cell[w][v]), kCellShift, 16) * sizeof(uint2))));
          }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int w = 0; w < kBatch; w++)
#pragma unroll
          for (int v = 0; v < VEC; v++) {
            bn[w][v] = table_start(entry[w][v], cell[w][v]);
            at[w][v] = (c_prop[v] + bn[w][v] * static_cast<int>(sizeof(T))) & table_occupied(entry[w][v], cell[w][v]);
          }
      }
      // Where the bit of a value's cell is not set (seven of eight cells) the start is the bin: such lanes read the +inf entries
      // at the front, all at one address, and the LDS serves the few others without many conflicts. Else the table gives a proposal at or before the value's bin; the proposals from there on
      // are ascending, so the bin is that start plus the number of proposals below the value.
      // Three of them are compared at once, without a branch; the (rare) lanes that saw three
      // smaller proposals look at four more, and then finish with a binary search.
      bool more = false;
      {
        T probe[kBatch][VEC][3];
#pragma unroll
        for (int w = 0; w < kBatch; w++)
#pragma unroll
          for (int v = 0; v < VEC; v++)
#pragma unroll
            for (int i = 0; i < 3; i++) probe[w][v][i] = reinterpret_cast<const T*>(smem_raw + at[w][v])[i];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int w = 0; w < kBatch; w++)
#pragma unroll
          for (int v = 0; v < VEC; v++) {
            const T x = xs[w][v];
            bn[w][v] += probe[w][v][0] < x ? 1 : 0;
            bn[w][v] += probe[w][v][1] < x ? 1 : 0;
            bn[w][v] += probe[w][v][2] < x ? 1 : 0;
            more = more || probe[w][v][2] < x;
          }
      }
      if (__any(more)) {
#pragma unroll
        for (int w = 0; w < kBatch; w++)
#pragma unroll
          for (int v = 0; v < VEC; v++) {
            // smaller proposals end at bn: the one before it is smaller whether three were or fewer
            const T x   = xs[w][v];
            const T* pp = reinterpret_cast<const T*>(smem_raw + c_prop[v]) + bn[w][v];
            if (!__any(pp[0] < x)) continue;
            const int c2 = (pp[0] < x ? 1 : 0) + (pp[1] < x ? 1 : 0) + (pp[2] < x ? 1 : 0) + (pp[3] < x ? 1 : 0);
            bn[w][v] += c2;
            if (__any(c2 == 4)) {
              const int f    = kRagged ? min(fb + v, f1 - 1) : fb + v;
              const int left = c2 == 4 ? a.row_pointers[f + 1] - a.row_pointers[f] - bn[w][v] : 0;
              bn[w][v] += count_less(pp + 4, left, x, a.search_steps);
            }
          }
      }
#pragma unroll
      for (int w = 0; w < kBatch; w++) {
        constexpr int kInWord = 4 / sizeof(BinT);
        const int u = u0 + w;
        uint32_t words[2] = {0u, 0u};
#pragma unroll
        for (int v = 0; v < VEC; v++) {
          const int b = kRagged && v >= mine ? 0 : bn[w][v];
          words[v / kInWord] |= static_cast<uint32_t>(b) << (8 * sizeof(BinT) * (v % kInWord));
        }
        if constexpr (kShared) {
          pair_of[u] = q_c[u % kAhead];
#pragma unroll
          for (int k = 0; k < kWords; k++) words[k] = kind == 0 ? words[k] : 0u;
        } else if constexpr (!kByByte) {
          uint32_t pair[2];
          if constexpr (kWords == 2) {
            pair[0] = static_cast<uint32_t>(q_c[u % kAhead].x);
            pair[1] = static_cast<uint32_t>(q_c[u % kAhead].y);
          } else {
            pair[0] = pair[1] = static_cast<uint32_t>(q_c[u % kAhead]);
          }
#pragma unroll
          for (int k = 0; k < kWords; k++) words[k] = kind == 0 ? words[k] : (pair[k] & pair_mask);
        }
#pragma unroll
        for (int k = 0; k < kWords; k++) own[u][k] = words[k];
        x_c[u % kAhead] = load_row(x_off + (u + kAhead) * x_step);
        if constexpr (!kByByte) q_c[u % kAhead] = load_pair(q_off + (u + kAhead) * q_step);
      }
    }
    const int left = n_local - first - rsub;  // row u of the pass exists if u * rpp < left
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
      if (u * a.rpp >= left) continue;  // (the same for the lanes of a row)
      unsigned char* const to = b_chunk + (b_off + u * b_step);
      if constexpr (kShared) {
        const uint32_t w0 = own[u][0], w1 = kWords == 2 ? own[u][kWords - 1] : 0u;
        const uint32_t p0 = static_cast<uint32_t>(pair_of[u].x), p1 = static_cast<uint32_t>(pair_of[u].y);
        if (a.share == 1) {
          *reinterpret_cast<uint4*>(to)      = make_uint4(w0, w1, 0u, 0u);
          *reinterpret_cast<uint4*>(to + 16) = make_uint4(0u, 0u, p0, p1);
        } else if (a.share == 2) {
          const uint32_t o0 = quad_lane<0xb1>(w0), o1 = kWords == 2 ? quad_lane<0xb1>(w1) : 0u;  // of the other lane
          const uint4 bins  = kOwn == 8   ? make_uint4(w0, w1, o0, o1)
                              : kOwn == 4 ? make_uint4(w0, o0, 0u, 0u)
                                          : make_uint4(w0 | o0 << (8 * kOwn % 32), 0u, 0u, 0u);
          *reinterpret_cast<uint4*>(to) = to_off == 0 ? bins : make_uint4(0u, 0u, p0, p1);
        } else {
          const uint32_t b0 = quad_lane<0 + 4 * 2>(w0), b1 = quad_lane<1 + 4 * 3>(w0);  // lane 0: of lanes 0 and 1, lane 1: of lanes 2 and 3
          const uint2 last  = to_off == 24 ? make_uint2(p0, p1) : make_uint2(0u, 0u);
          *reinterpret_cast<uint2*>(to) = to_off < 16 ? make_uint2(b0, b1) : last;
        }
      } else if constexpr (kByByte) {
        if constexpr (kOwn == 2)
          *reinterpret_cast<uint16_t*>(to) = static_cast<uint16_t>(own[u][0]);
        else
          *to = static_cast<unsigned char>(own[u][0]);
        for (int i = kOwn; i < t_zero; i++) to[i] = 0;
        if (t_pair >= 0) *reinterpret_cast<int2*>(to + t_pair) = load_pair(q_off + u * q_step);
      } else if constexpr (kWords == 2) {
        *reinterpret_cast<uint2*>(to) = make_uint2(own[u][0], own[u][1]);
      } else {
        *reinterpret_cast<uint32_t*>(to) = own[u][0];
      }
    }
    x_off += kUnroll * x_step;
    b_off += kUnroll * b_step;
    q_off += kUnroll * q_step;
  };
  auto walk = [&](auto bent_cells) {
    if (n_local <= 0) return;
    Vec x_c[kAhead];
    Pair q_c[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; u++) {
      x_c[u] = load_row(x_off + u * x_step);
      if constexpr (!kByByte) q_c[u] = load_pair(q_off + u * q_step);
    }
    for (int first = 0; first < n_local; first += pass_rows) search_pass(bent_cells, first, x_c, q_c);
  };
  if (bent)
    walk(std::true_type{});
  else
    walk(std::false_type{});
}

// A lane's kPer bins of a row whose 64 record bytes the aligned group of four lanes holds, 16 bytes each: lane l's from
// byte kPer * l on, of which up to three words lie with the lane before (all four have to be active).
// m: how many. perm: the byte order of the results, which are the bins 0..3, 4..7, 8..11 (and, 16 of them, 12..15) of the lane,
// each four turned by its row's place in the quarter wave; the last word of 13 or 14 holds the others from byte
// kPer * l modulo 4 on, unturned.
template <int kPer>
__device__ __forceinline__ uint4 spread_bins(const uint4& w, int m, uint32_t perm)
{
  static_assert(kPer == 12 || kPer == 13 || kPer == 14 || kPer == 16, "a lane's bins then lie in four words, the first not before the lane before");
  auto turn = [&](uint32_t hi, uint32_t lo) { return __builtin_amdgcn_perm(hi, lo, perm); };
  if constexpr (kPer == 16) return make_uint4(turn(w.x, w.x), turn(w.y, w.y), turn(w.z, w.z), turn(w.w, w.w));
  auto before = [](uint32_t v) { return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), 0x90, 0xf, 0xf, true)); };  // lanes 0, 0, 1, 2
  const uint32_t p1 = before(w.y), p2 = before(w.z), p3 = before(w.w);
  const bool one = (m & 1) != 0, two = (m & 2) != 0;
  const uint32_t t0 = one ? p1 : p2, t1 = one ? p2 : p3, t2 = one ? p3 : w.x, t3 = one ? w.x : w.y, t4 = one ? w.y : w.z,
                 t5 = one ? w.z : w.w;
  const uint32_t o0 = two ? t0 : t2, o1 = two ? t1 : t3, o2 = two ? t2 : t4, o3 = two ? t3 : t5;
  return make_uint4(turn(o1, o0), turn(o2, o1), turn(o3, o2), o3);
}

// Histogram of one level from the cached bins: a lane loads BV cached bins of its
// row with one load and only accumulates.
template <typename BinT, int BV>
struct BinVec;
template <>
struct BinVec<uint16_t, 4> {
  using type = uint2;
};
template <>
struct BinVec<uint8_t, 16> {
  using type = uint4;
};

template <typename BinT, int BV>
__device__ inline void unpack_bins(const typename BinVec<BinT, BV>::type& w, int (&out)[BV])
{
  if constexpr (BV == 16) {
    const uint32_t q[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
      out[4 * i + 0] = q[i] & 0xff;
      out[4 * i + 1] = (q[i] >> 8) & 0xff;
      out[4 * i + 2] = (q[i] >> 16) & 0xff;
      out[4 * i + 3] = q[i] >> 24;
    }
  } else {
    out[0] = w.x & 0xffff;
    out[1] = w.x >> 16;
    out[2] = w.y & 0xffff;
    out[3] = w.y >> 16;
  }
}

struct BinnedArgs {
  TileWalk w;
  const RecInfo* rec;  // [groups]
  int K;
  const int32_t* row_pointers;
  const int32_t* groups;
  HistView hist;
  Stripes stripes;  // layout of the LDS sub-histogram
  int lanes;        // lanes per row for every group of the launch; 0: as many as the group's own features need
  int sync_every;   // tiles between two meeting points of the root launch's workgroups
};

// The 16 bytes of `w` rotated down by t bytes: byte v of the result is byte (v + t) mod 16 of w.
__device__ __forceinline__ uint4 rotate_bytes(const uint4& w, int t)
{
  const bool r1 = (t & 4) != 0, r2 = (t & 8) != 0;
  const uint32_t x1 = r1 ? w.y : w.x, y1 = r1 ? w.z : w.y, z1 = r1 ? w.w : w.z, w1 = r1 ? w.x : w.w;
  const uint32_t x2 = r2 ? z1 : x1, y2 = r2 ? w1 : y1, z2 = r2 ? x1 : z1, w2 = r2 ? y1 : w1;
  const uint32_t b = static_cast<uint32_t>(t) & 3u;
  return make_uint4(__builtin_amdgcn_alignbyte(y2, x2, b), __builtin_amdgcn_alignbyte(z2, y2, b),
                    __builtin_amdgcn_alignbyte(w2, z2, b), __builtin_amdgcn_alignbyte(x2, w2, b));
}

// The value that lane kLane of the caller's aligned group of four lanes holds (all four have to be active).
template <int kLane>
__device__ __forceinline__ int quad_lane(int v)
{
  return __builtin_amdgcn_update_dpp(0, v, kLane * 0x55, 0xf, 0xf, false);
}

// 4 x 4 byte transpose: input word r is row r and its byte b is feature b; output word b holds
// feature b of rows 0..3.
__device__ __forceinline__ void turn_bytes(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3, uint32_t (&out)[4])
{
  const uint32_t a = __builtin_amdgcn_perm(w1, w0, 0x05010400u);
  const uint32_t b = __builtin_amdgcn_perm(w1, w0, 0x07030602u);
  const uint32_t c = __builtin_amdgcn_perm(w3, w2, 0x05010400u);
  const uint32_t d = __builtin_amdgcn_perm(w3, w2, 0x07030602u);
  out[0]           = __builtin_amdgcn_perm(c, a, 0x05040100u);
  out[1]           = __builtin_amdgcn_perm(c, a, 0x07060302u);
  out[2]           = __builtin_amdgcn_perm(d, b, 0x05040100u);
  out[3]           = __builtin_amdgcn_perm(d, b, 0x07060302u);
}

// kEmbed: the records carry the packed (grad, hess) of their row (single-output trees);
// otherwise the pair of (row, output) is gathered from qgh.
// kRoot: the launch for the root, whose rows are still in their original order. A lane then
// takes four consecutive rows per tile and, besides accumulating, stores their bins feature by
// feature into bins_t ([feature][row]), which the position updates read: the feature-major copy
// costs no second pass over the cache.
// kStriped (one-byte bins): the LDS sub-histogram is striped (see Stripes) and every lane takes the
// 16 bins of a row in its own rotated order.
// kPer (striped; 0: not): every group of the launch has four lanes per row (and a lane four rows per tile), so the lanes of a
// row are an aligned group of four. They share the row's bins evenly, kPer each, instead of 16, 16, 16 and what is left, and an
// atomic is one vector instruction beside itself (see Stripes): 2,000,000 x 200, 8 outputs: 4.4 vector instructions an atomic
// at 13 bins a lane, 6.7 when its address took three. What all four of them need one of them loads and hands round with a
// cross-lane move: a vector memory instruction costs by the cache lines it touches and holds registers until it
// returns. Below the root lane u of the four loads the position of the tile's row u and, with several outputs, its
// gradient pair. With one output (kQuad) the record is the four lanes' 64 bytes and its last 8 the pair: it comes out of
// the fourth lane's bins.
constexpr int kStripeMaxW = 256;  // widest group the striped layout serves, in features
__host__ __device__ constexpr size_t spread_hist_bytes(int bins) { return 65536 + static_cast<size_t>(bins) * 256; }
constexpr size_t kSpreadMore = (static_cast<size_t>(kTileWindow) * 16 + 64 * 4 + 4 + 15) / 16 * 16;  // tile window, offsets, slot

template <typename BinT, int BV, bool kEmbed, bool kRoot, bool kStriped, int kPer>
__global__ void __launch_bounds__(kHistThreads)
  binned_histogram_kernel(BinnedArgs a, LBT_WALK_PARAMS, const unsigned char* __restrict__ cache,
                          const int2* __restrict__ qgh, BinT* __restrict__ bins_t, int64_t bins_t_stride,
                          int32_t* pair_sync, PartialSink sink)
{
  static_assert(!kStriped || BV == 16, "the striped layout is built for lanes that hold 16 one-byte bins");
  static_assert(kPer == 0 || kStriped, "four lanes per row: a mode of the striped kernel");
  constexpr bool kQuad = kPer > 0 && kEmbed;
  using Word = typename BinVec<BinT, BV>::type;
  constexpr int kRows = kRoot ? 4 : (BV == 16 ? kBinnedUnroll / 2 : kBinnedUnroll);  // rows per lane and tile
  static_assert(kPer == 0 || kRows == 4, "each of a row's four lanes asks for one of the tile's four rows");
  extern __shared__ __align__(16) unsigned char smem_raw[];  // 16-byte aligned whatever static LDS precedes it
  int* s_slot;
  int* s_off;  // striped: first bin of every feature in the group's run of bins
  int4* s_tile_window;
  if constexpr (kPer > 0) {
    // behind the sub-histogram, which has to begin at address 0: no static LDS (the launch looks)
    s_tile_window = reinterpret_cast<int4*>(smem_raw + spread_hist_bytes(a.stripes.bins));
    s_off         = reinterpret_cast<int*>(s_tile_window + kTileWindow);
    s_slot        = s_off + 64;
  } else {
    __shared__ int slot_word;
    __shared__ int offsets[kStriped ? kStripeMaxW : 1];
    __shared__ int4 window[kTileWindow];
    s_slot        = &slot_word;
    s_off         = offsets;
    s_tile_window = window;
  }
  const TileWalk& w = a.w;
  const int xcd   = blockIdx.x & 7;
  const int slot  = blockIdx.x >> 3;
  const int gk    = slot % w.n_gk;
  const int chunk = (slot / w.n_gk) * 8 + xcd;
  const int group = gk / a.K;
  const int k     = gk % a.K;
  const int f0 = a.groups[group], f1 = a.groups[group + 1];
  const int gs   = f1 - f0;
  const int bin0 = a.row_pointers[f0];
  const int nb   = a.row_pointers[f1] - bin0;
  unsigned long long* s_hist = reinterpret_cast<unsigned long long*>(smem_raw);
  // `per` as it was compiled: read from the arguments, every variant carries all layouts' code and gives registers for it. The seven
  // launches below the root, us: 20,000,000 x 24 1433 before there was a `per`, 1466 with it from the arguments, now 1426;
  // 2,200,000 x 20 with 8 outputs 681, 705, 681.
  const Stripes st{a.stripes.log_w, a.stripes.bins, kPer};
  if constexpr (kStriped) {
    for (int i = threadIdx.x; i < st.words(); i += kHistThreads) s_hist[st.place(i)] = 0;
    for (int i = threadIdx.x; i < (1 << st.log_w); i += kHistThreads)
      s_off[i] = i < gs ? a.row_pointers[f0 + i] - bin0 : 0;
  } else {
    // behind the group's bins every lane owns a spare slot that takes the adds of its features
    // past the group end (never read; private, so these adds do not collide)
    for (int i = threadIdx.x; i < nb + kHistThreads; i += kHistThreads) s_hist[i] = 0;
  }

  const RecInfo ri        = a.rec[group];
  // With the same number of lanes per row in every group (a narrower group's last lanes then add the
  // zero bytes of its record's padding to columns that nothing reads) the workgroups of the groups
  // that walk the same rows run the same instructions tile after tile and stay side by side
  // without waiting for each other: the cache line that holds a row's records is then still in the
  // L2 when the second of them asks for it.
  const int lanes_per_row = kPer > 0 ? 4 : (a.lanes > 0 ? a.lanes : (gs + BV - 1) / BV);
  const int lr            = threadIdx.x % lanes_per_row;
  const int rsub          = threadIdx.x / lanes_per_row;
  const bool active       = rsub < w.rpp;
  const int fl            = lr * BV;
  const int my_off        = lr * static_cast<int>(sizeof(Word));
  const unsigned char* const my_rec = cache + ri.base;
  const int64_t stride              = ri.stride;
  // the gradient pair may share the last 16 bytes a lane loads as bins: that lane blanks them
  const bool strip = kEmbed && BV == 16 && ri.q_off >= my_off && ri.q_off < my_off + static_cast<int>(sizeof(Word));
  const int nv = min(BV, max(0, gs - fl));  // features this lane really has
  // packed layout: first word of every feature of the lane. Striped: the lane's step v works on its
  // byte (v + rot) mod 16; c_base[v] is the byte offset of that feature's column in the LDS array
  // and bit v of `has` says whether the lane has that feature.
  const int rot = threadIdx.x & 15;
  unsigned has  = 0;
  int c_base[BV];
#pragma unroll
  for (int v = 0; v < BV; v++) {
    if constexpr (kStriped) {
      const int o = (v + rot) & 15;
      c_base[v]   = (fl + o) * 8;
      has |= o < nv ? (1u << v) : 0u;
    } else {
      c_base[v] = fl + v < gs ? a.row_pointers[f0 + fl + v] - bin0 : nb + threadIdx.x;
    }
  }
  // The bytes of a lane's 16 that lie past the group's last feature are zeros (record padding, the
  // blanked gradient pair): added as they are, they would all fall into bin 0 of their column, and
  // the lanes that hold the same column in the four quarters of a wave (thread t, t + 16, ...)
  // would hit one address at every step, which the LDS serialises (3 cycles of
  // SQ_LDS_ADDR_CONFLICT per atomic, one more cycle per wave-level atomic in a kernel that does
  // nothing else; 1 % of these launches, where the LDS is busy less than half of the time). Each
  // quarter sends them to a bin of its own instead; nothing reads those columns.
  uint4 pad_or = make_uint4(0u, 0u, 0u, 0u);
  if constexpr (kStriped) {
    const uint32_t q4 = min((static_cast<uint32_t>(threadIdx.x) >> 4) & 3u, static_cast<uint32_t>(max(st.bins, 1) - 1));
    uint32_t pw[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int j = 0; j < 16; j++)
      if (fl + j >= gs) pw[j >> 2] |= q4 << (8 * (j & 3));
    pad_or = make_uint4(pw[0], pw[1], pw[2], pw[3]);
  }
  const int stripe_shift = st.log_w + 3;  // a bin's row of the striped array, in bytes
  // kPer: the feature, in the group, that the lane takes at step v, and its column (see Stripes); qr: the row's place in
  // the quarter wave
  const int qr = (threadIdx.x >> 2) & 3;
  auto spread_feature = [&](int v) {
    const int c = v < 12 || kPer == 16 ? 4 * (v >> 2) + ((v + qr) & 3) : (kPer == 13 ? 12 : 12 + ((qr & 1) ^ (v - 12)));
    return kPer * lr + c;
  };
  const int words_before     = 4 * lr - ((kPer * lr) >> 2);
  const uint32_t bytes_ahead = static_cast<uint32_t>(kPer * lr) & 3u;
  uint32_t spread_perm       = 0;
#pragma unroll
  for (int j = 0; j < 4; j++) spread_perm |= (bytes_ahead + static_cast<uint32_t>((j + qr) & 3)) << (8 * j);
  // bytes of the words' addresses: the low ones of the steps of a group of four (a 128-byte block further in the second
  // and fourth group, which the instruction's offset adds) and, for columns from 32 on, the 1 of the 64 KB; those of the
  // features beyond 12
  uint32_t low_of = 0, half_of[2] = {1u << 16, 1u << 16}, beyond[2] = {0, 0};
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const uint32_t low = 8u * static_cast<uint32_t>(4 * ((j + qr) & 3) + lr);
    low_of |= low << (8 * j);
    if (j < 3) half_of[0] |= low << (8 * (j == 2 ? 3 : j));
    else half_of[1] |= low;
  }
#pragma unroll
  for (int e = 0; e < 2; e++) {
    const int x       = kPer == 13 ? 0 : (qr & 1) ^ e;  // which of the lane's features beyond 12
    const int column  = lr + (kPer == 13 ? 4 * qr : 8 * x + 4 * (qr >> 1));
    half_of[1] |= static_cast<uint32_t>(128 + 8 * column) << (8 * (e == 0 ? 1 : 3));
    beyond[e] = 0x0c020000u | ((4u + bytes_ahead + static_cast<uint32_t>(x)) << 8) | (e == 0 ? 1u : 3u);
  }
  using LdsWord = __attribute__((address_space(3))) unsigned long long;
  auto add_spread = [&](const uint4& bins, unsigned long long packed) {
    auto add = [&](uint32_t address, int block) {
      __hip_atomic_fetch_add(reinterpret_cast<LdsWord*>(static_cast<uintptr_t>(address)) + 16 * block, packed, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    const uint32_t q[4] = {bins.x, bins.y, bins.z, bins.w};
#pragma unroll
    for (int v = 0; v < kPer; v++) {
      const uint32_t j = static_cast<uint32_t>(v) & 3u;
      if (v < 8)
        add(__builtin_amdgcn_perm(q[v >> 2], low_of, 0x0c0c0000u | ((4u + j) << 8) | j), v >> 2);
      else if (v < 12 || kPer == 16)
        add(__builtin_amdgcn_perm(q[v >> 2], half_of[j == 3u], 0x0c020000u | ((4u + j) << 8) | (j == 3u ? 0u : (j == 2u ? 3u : j))), (v >> 2) - 2);
      else
        add(__builtin_amdgcn_perm(q[3], half_of[1], beyond[v - 12]), 0);
    }
  };
  const unsigned long long max_abs = qstats[0];
  const int n_tiles = meta->n_tiles;
  const int t_begin = static_cast<int>(static_cast<int64_t>(n_tiles) * chunk / w.n_chunks);
  const int t_end   = static_cast<int>(static_cast<int64_t>(n_tiles) * (chunk + 1) / w.n_chunks);
  int cur_node           = -1;
  unsigned long long acc = 0;
  // rows of cur_node that this workgroup has taken, and how many the node has: when they
  // agree at the end of the node, its bins belong to this workgroup alone. Not when single
  // tiles may go to the histogram directly (huge gradients), which other workgroups may do too,
  // and not when a part of the node has left the LDS before its end (node_flushed): without a
  // free slot that part was added to the histogram with atomics during this launch, and a plain
  // store of the rest would overwrite it.
  int node_rows = 0, node_total = 0;
  bool node_flushed = false;
  const bool owners = static_cast<unsigned long long>(w.tile_rows) * max_abs <= 2147483647ULL;
  __syncthreads();

  // positions a lane keeps per tile: with kQuad only that of the row with its own number among the four lanes
  constexpr int kPos = kPer > 0 && !kRoot ? 1 : kRows;
  auto load_rows = [&](const Tile& t, int (&row)[kPos]) -> unsigned {
    unsigned valid = 0;
    if constexpr (kPer > 0 && !kRoot) {
      const int mine = t.r0 + rsub + lr * w.rpp;
      row[0]         = positions[mine < t.r1 ? mine : t.r0];
#pragma unroll
      for (int u = 0; u < kRows; u++) valid |= t.r0 + rsub + u * w.rpp < t.r1 ? (1u << u) : 0u;
      return valid;
    }
#pragma unroll
    for (int u = 0; u < kRows; u++) {
      const int rr  = kRoot ? t.r0 + kRows * rsub + u : t.r0 + rsub + u * w.rpp;
      const bool ok = active && rr < t.r1;
      if constexpr (kRoot)
        row[u] = ok ? rr : t.r0;  // the order is still the identity: sorted index == row
      else
        row[u] = positions[ok ? rr : t.r0];
      valid |= ok ? (1u << u) : 0u;
    }
    return valid;
  };
  // gradient pairs a lane loads per tile: none (one unused slot) when they come out of the fourth lane's bins, one for its own
  // row where the lanes hand them round
  constexpr int kPairs = kQuad || (kPer > 0 && !kRoot) ? 1 : kRows;
  auto load_data = [&](const int (&row)[kPos], Word (&bw)[kRows], int2 (&q)[kPairs]) {
    int rws[kRows];
    if constexpr (kPer > 0 && !kRoot && !kEmbed) q[0] = qgh[static_cast<int64_t>(row[0]) * a.K + k];
    if constexpr (kPer > 0 && !kRoot) {
      rws[0] = quad_lane<0>(row[0]);
      rws[1] = quad_lane<1>(row[0]);
      rws[2] = quad_lane<2>(row[0]);
      rws[3] = quad_lane<3>(row[0]);
    } else {
#pragma unroll
      for (int u = 0; u < kRows; u++) rws[u] = row[u];
    }
#pragma unroll
    for (int u = 0; u < kRows; u++) {
      const int64_t rw          = rws[u];
      const unsigned char* recp = my_rec + rw * stride;
      bw[u]                     = *reinterpret_cast<const Word*>(recp + my_off);
      if constexpr (kQuad || (kPer > 0 && !kRoot)) {
      } else if constexpr (kEmbed) {
        q[u] = *reinterpret_cast<const int2*>(recp + ri.q_off);
      } else {
        q[u] = qgh[rw * a.K + k];
      }
    }
  };

  TileWindow win{s_tile_window, tiles, 0, t_end};
  win.fill(t_begin);
  Tile tc{}, tn{}, tnn{};
  int row_c[kPos], row_n[kPos], row_nn[kPos];
  Word b_c[kRows], b_n[kRows];
  int2 q_c[kPairs], q_n[kPairs];
  unsigned valid_c = 0, valid_n = 0, valid_nn = 0;
#pragma unroll
  for (int u = 0; u < kPos; u++) row_c[u] = row_n[u] = row_nn[u] = 0;
#pragma unroll
  for (int u = 0; u < kPairs; u++) q_c[u] = q_n[u] = make_int2(0, 0);
  if (t_begin < t_end) {
    tc      = win.get(t_begin);
    valid_c = load_rows(tc, row_c);
    load_data(row_c, b_c, q_c);
  }
  if (t_begin + 1 < t_end) {
    tn      = win.get(t_begin + 1);
    valid_n = load_rows(tn, row_n);
  }

  for (int tile = t_begin; tile < t_end; tile++) {
    if constexpr (kRoot) {
      // The workgroups of the feature groups (and outputs) that walk the same rows read the
      // same cache lines (a row's records share a line). Every kPairSyncTiles tiles each one
      // counts itself in and gives the others a bounded time to catch up, so that the line one
      // of them fetched is still in the L2 when the next one asks for it. Only a hint: after
      // kPairSyncSpins polls a workgroup goes on regardless.
      const int done = tile - t_begin;
      if (pair_sync != nullptr && done > 0 && done % a.sync_every == 0) {
        if (threadIdx.x == 0) {
          const int want = done / a.sync_every * w.n_gk;
          __hip_atomic_fetch_add(pair_sync + chunk, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          for (int spin = 0; spin < kPairSyncSpins; spin++) {
            if (__hip_atomic_load(pair_sync + chunk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= want) break;
            __builtin_amdgcn_s_sleep(32);
          }
        }
        __syncthreads();
      }
    }
    // kTurned: the tile's bins are taken out of the registers they were loaded into before the next tile's are asked for, so
    // that nothing is moved at the end of the turn
    constexpr bool kTurned = kPer > 0 && !kRoot;
    Word bins[kTurned ? kRows : 1];
    int2 pairs[kTurned ? kRows : 1];
    if constexpr (kTurned) {
      if constexpr (!kQuad) {
        pairs[0] = make_int2(quad_lane<0>(q_c[0].x), quad_lane<0>(q_c[0].y));
        pairs[1] = make_int2(quad_lane<1>(q_c[0].x), quad_lane<1>(q_c[0].y));
        pairs[2] = make_int2(quad_lane<2>(q_c[0].x), quad_lane<2>(q_c[0].y));
        pairs[3] = make_int2(quad_lane<3>(q_c[0].x), quad_lane<3>(q_c[0].y));
      }
#pragma unroll
      for (int u = 0; u < kRows; u++) {
        Word w = b_c[u];
        if constexpr (kQuad) {
          pairs[u] = make_int2(quad_lane<3>(static_cast<int>(w.z)), quad_lane<3>(static_cast<int>(w.w)));
          w.z      = strip ? 0u : w.z;
          w.w      = strip ? 0u : w.w;
        }
        w.x |= pad_or.x;
        w.y |= pad_or.y;
        w.z |= pad_or.z;
        w.w |= pad_or.w;
        bins[u] = spread_bins<kPer>(w, words_before, spread_perm);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (tile + 1 < t_end) load_data(row_n, b_c, q_c);
    } else {
      if (tile + 1 < t_end) load_data(row_n, b_n, q_n);
    }
    if (tile + 2 < t_end) {
      tnn      = win.get(tile + 2);
      valid_nn = load_rows(tnn, row_nn);
    }
    const int nrows   = tc.r1 - tc.r0;
    const bool direct = tc.seg_rows < kSmallNodeRows ||
                        static_cast<unsigned long long>(nrows) * max_abs > 2147483647ULL;
    if (!direct) {
      if (tc.node != cur_node || (acc + nrows) * max_abs > 2147483647ULL) {
        __syncthreads();
        if (cur_node >= 0)
          park_sub_histogram(s_hist, nb, a.hist.at(cur_node, k, bin0), sink,
                             (cur_node - w.level_first - w.j0) * w.n_gk + gk, s_slot,
                             owners && tc.node != cur_node && !node_flushed && node_rows == node_total, st, s_off,
                             gs);
        __syncthreads();
        node_flushed = tc.node == cur_node;
        if (tc.node != cur_node) {
          node_rows  = 0;
          node_total = tc.seg_rows;
        }
        cur_node = tc.node;
        acc      = 0;
      }
      acc += nrows;
      node_rows += nrows;
    }
    int2 qv[kRows];
#pragma unroll
    for (int u = 0; u < kRows; u++) {
      if constexpr (kTurned)
        qv[u] = pairs[u];
      else if constexpr (kQuad)
        qv[u] = make_int2(quad_lane<3>(static_cast<int>(b_c[u].z)), quad_lane<3>(static_cast<int>(b_c[u].w)));
      else
        qv[u] = q_c[u];
    }
    if constexpr (kEmbed && BV == 16 && !kTurned) {
#pragma unroll
      for (int u = 0; u < kRows; u++) {
        b_c[u].z = strip ? 0u : b_c[u].z;
        b_c[u].w = strip ? 0u : b_c[u].w;
      }
    }
    if constexpr (kRoot) {
      // feature-major copy; rows past the end of the tile hold the bins of the tile's first row,
      // and bins_t is padded to whole groups of rows
      // the workgroups of the K outputs read the same records: they share the copy between them,
      // output k takes every K-th piece of four features (one output's workgroups alone would
      // write K times as long as the others and hold the launch up)
      if (valid_c & 1u) {
        const int64_t row0 = row_c[0];
        if constexpr (BV == 16) {
          BinT* dst = bins_t + static_cast<int64_t>(f0 + fl) * bins_t_stride + row0;
          auto put  = [&](int i, uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3) {
            if ((lr * 4 + i) % a.K != k) {
              dst += 4 * bins_t_stride;
              return;
            }
            uint32_t o[4];
            turn_bytes(w0, w1, w2, w3, o);
#pragma unroll
            for (int j = 0; j < 4; j++) {
              if (fl + 4 * i + j < gs) *reinterpret_cast<uint32_t*>(dst) = o[j];
              dst += bins_t_stride;
            }
          };
          put(0, b_c[0].x, b_c[1].x, b_c[2].x, b_c[3].x);
          put(1, b_c[0].y, b_c[1].y, b_c[2].y, b_c[3].y);
          put(2, b_c[0].z, b_c[1].z, b_c[2].z, b_c[3].z);
          put(3, b_c[0].w, b_c[1].w, b_c[2].w, b_c[3].w);
        } else {
          // four two-byte bins per row
          const uint32_t lo[4] = {b_c[0].x, b_c[1].x, b_c[2].x, b_c[3].x};
          const uint32_t hi[4] = {b_c[0].y, b_c[1].y, b_c[2].y, b_c[3].y};
          uint2 o[4];
          o[0] = make_uint2((lo[0] & 0xffffu) | (lo[1] << 16), (lo[2] & 0xffffu) | (lo[3] << 16));
          o[1] = make_uint2((lo[0] >> 16) | (lo[1] & 0xffff0000u), (lo[2] >> 16) | (lo[3] & 0xffff0000u));
          o[2] = make_uint2((hi[0] & 0xffffu) | (hi[1] << 16), (hi[2] & 0xffffu) | (hi[3] << 16));
          o[3] = make_uint2((hi[0] >> 16) | (hi[1] & 0xffff0000u), (hi[2] >> 16) | (hi[3] & 0xffff0000u));
#pragma unroll
          for (int v = 0; v < 4; v++)
            if (fl + v < gs && (lr * 4 + v) % a.K == k)
              *reinterpret_cast<uint2*>(bins_t + static_cast<int64_t>(f0 + fl + v) * bins_t_stride + row0) = o[v];
        }
      }
    }
    if constexpr (kStriped && !kTurned) {
      // from here on a lane's bins stand in its own order (the feature-major copy above took them as loaded)
#pragma unroll
      for (int u = 0; u < kRows; u++) {
        b_c[u].x |= pad_or.x;
        b_c[u].y |= pad_or.y;
        b_c[u].z |= pad_or.z;
        b_c[u].w |= pad_or.w;
        if constexpr (kPer > 0)
          b_c[u] = spread_bins<kPer>(b_c[u], words_before, spread_perm);
        else
          b_c[u] = rotate_bytes(b_c[u], rot);
      }
    }
    if (!direct) {
#pragma unroll
      for (int u = 0; u < kRows; u++) {
        if (valid_c & (1u << u)) {
          const unsigned long long packed = pack_pair(qv[u].x, qv[u].y);
          if constexpr (kPer > 0) {
            if constexpr (kTurned)
              add_spread(bins[u], packed);
            else
              add_spread(b_c[u], packed);
            continue;
          }
          int rel[BV];
          unpack_bins<BinT, BV>(b_c[u], rel);
#pragma unroll
          // a lane whose 16 bins reach past the group end leaves those out: an atomic costs by
          // the lanes that take part in it
          for (int v = 0; v < BV; v++) {
            if constexpr (kStriped) {
              // no test per bin: the bytes past the group's last feature are zeros and belong to columns of
              // the array that no feature owns and no merge reads (an atomic costs by the instruction, not
              // by the lanes that take part, and a test costs two branches)
              atomicAdd(reinterpret_cast<unsigned long long*>(smem_raw + ((rel[v] << stripe_shift) + c_base[v])), packed);
            } else {
              if (v < nv) atomicAdd(&s_hist[c_base[v] + rel[v]], packed);
            }
          }
        }
      }
    } else {
      I64Pair* gdst = a.hist.at(tc.node, k, bin0);
#pragma unroll
      for (int u = 0; u < kRows; u++) {
        if (valid_c & (1u << u)) {
          int rel[BV];
          if constexpr (kTurned)
            unpack_bins<BinT, BV>(bins[u], rel);
          else
            unpack_bins<BinT, BV>(b_c[u], rel);
          if constexpr (kPer == 13 || kPer == 14) {
            // the bins from 12 on stand as they were loaded, the turned ones as the steps take them
            const uint32_t last = kTurned ? bins[kTurned ? u : 0].w : b_c[u].w;
#pragma unroll
            for (int v = 12; v < kPer; v++)
              rel[v] = static_cast<int>((last >> (8 * (bytes_ahead + static_cast<uint32_t>(spread_feature(v) - kPer * lr - 12)))) & 0xffu);
          }
#pragma unroll
          for (int v = 0; v < (kPer > 0 ? kPer : BV); v++) {
            bool mine;
            int bin;
            if constexpr (kPer > 0) {
              const int f = spread_feature(v);
              mine = f < gs;
              bin  = mine ? s_off[f] + rel[v] : 0;
            } else if constexpr (kStriped) {
              mine = (has & (1u << v)) != 0;
              bin  = mine ? s_off[c_base[v] >> 3] + rel[v] : 0;
            } else {
              mine = fl + v < gs;
              bin  = c_base[v] + rel[v];
            }
            if (mine) {
              atomic_add_i64(&gdst[bin].grad, static_cast<int64_t>(qv[u].x));
              atomic_add_i64(&gdst[bin].hess, static_cast<int64_t>(qv[u].y));
            }
          }
        }
      }
    }
    tc      = tn;
    tn      = tnn;
    valid_c = valid_n;
    valid_n = valid_nn;
#pragma unroll
    for (int u = 0; u < kPos; u++) {
      row_c[u] = row_n[u];
      row_n[u] = row_nn[u];
    }
    if constexpr (!kTurned) {
#pragma unroll
      for (int u = 0; u < kRows; u++) b_c[u] = b_n[u];
#pragma unroll
      for (int u = 0; u < kPairs; u++) q_c[u] = q_n[u];
    }
  }
  __syncthreads();
  if (cur_node >= 0)
    park_sub_histogram(s_hist, nb, a.hist.at(cur_node, k, bin0), sink, (cur_node - w.level_first - w.j0) * w.n_gk + gk,
                       s_slot, owners && !node_flushed && node_rows == node_total, st, s_off, gs);
}

template <typename T, int VEC, bool kIdentityRows>
int launch_search(hipStream_t stream, const HistSetup& hs, const HistArgs<T>& a, const HistBatch& b, unsigned grid)
{
  static std::atomic<bool> attr_set[kMaxDevices] = {};
  LBT_TRY(allow_dynamic_lds(histogram_kernel<T, VEC, kIdentityRows>, kLdsBudget, attr_set));
  histogram_kernel<T, VEC, kIdentityRows><<<grid, kHistThreads, hs.lds_bytes, stream>>>(
    a, b.rows, hs.tiles, hs.meta, b.qstats, static_cast<const T*>(b.X), b.qgh);
  return LBT_OK;
}

template <typename T, int VEC>
int launch_search_rows(hipStream_t stream, const HistSetup& hs, const HistArgs<T>& a, const HistBatch& b,
                       unsigned grid, bool identity)
{
  if (identity) return launch_search<T, VEC, true>(stream, hs, a, b, grid);
  return launch_search<T, VEC, false>(stream, hs, a, b, grid);
}

template <typename T, int VEC, typename BinT, bool kRagged>
int launch_bin_rows(hipStream_t stream, const HistSetup& hs, const BinRowsArgs<T>& a, const HistBatch& b, unsigned grid)
{
  auto launch = [&](auto shared) -> int {
    constexpr bool kShared = decltype(shared)::value;
    static std::atomic<bool> attr_set[kMaxDevices] = {};
    LBT_TRY(allow_dynamic_lds(bin_rows_kernel<T, VEC, BinT, kRagged, kShared>, kLdsBudget, attr_set));
    bin_rows_kernel<T, VEC, BinT, kRagged, kShared><<<grid, kHistThreads, hs.lds_bytes, stream>>>(
      a, static_cast<const T*>(b.X), b.qgh, static_cast<BinT*>(hs.binned));
    return LBT_OK;
  };
  return hs.share > 0 ? launch(std::true_type{}) : launch(std::false_type{});
}

template <typename T, int VEC>
int launch_bin_rows_t(hipStream_t stream, const HistSetup& hs, const BinRowsArgs<T>& a, const HistBatch& b, unsigned grid)
{
  if constexpr (VEC > 1) {
    if (hs.ragged) {
      if (hs.bin_bytes == 1) return launch_bin_rows<T, VEC, uint8_t, true>(stream, hs, a, b, grid);
      return launch_bin_rows<T, VEC, uint16_t, true>(stream, hs, a, b, grid);
    }
  }
  if (hs.bin_bytes == 1) return launch_bin_rows<T, VEC, uint8_t, false>(stream, hs, a, b, grid);
  return launch_bin_rows<T, VEC, uint16_t, false>(stream, hs, a, b, grid);
}

template <typename BinT, int BV, bool kEmbed, bool kRoot, bool kStriped, int kPer = 0>
int launch_binned_as(hipStream_t stream, const HistSetup& hs, const BinnedArgs& a, const HistBatch& b, unsigned grid,
                     const PartialSink& sink)
{
  static std::atomic<bool> attr_set[kMaxDevices] = {};
  // the striped kernel without kPer keeps a table of feature offsets and its tile window in static LDS; with kPer they lie behind the
  // sub-histogram: neither asks for more than this
  LBT_TRY(allow_dynamic_lds(binned_histogram_kernel<BinT, BV, kEmbed, kRoot, kStriped, kPer>,
                            kStriped ? kLdsBudget - 8 * 1024 : kLdsBudget, attr_set));
  if constexpr (kPer > 0) {
    static std::atomic<int> static_lds{-1};
    if (static_lds.load(std::memory_order_relaxed) < 0) {
      hipFuncAttributes at{};
      LBT_HIP(hipFuncGetAttributes(&at, reinterpret_cast<const void*>(&binned_histogram_kernel<BinT, BV, kEmbed, kRoot, kStriped, kPer>)));
      static_lds.store(static_cast<int>(at.sharedSizeBytes), std::memory_order_relaxed);
    }
    LBT_REQUIRE(static_lds.load(std::memory_order_relaxed) == 0, "the sub-histogram has to begin at address 0 of the LDS");
  }
  binned_histogram_kernel<BinT, BV, kEmbed, kRoot, kStriped, kPer><<<grid, kHistThreads, hs.blds_bytes, stream>>>(
    a, b.rows, hs.tiles, hs.meta, b.qstats, static_cast<const unsigned char*>(hs.binned), b.qgh,
    static_cast<BinT*>(hs.bins_t), hs.bins_t_stride,
    // meeting points only between workgroups that run at the same time: one that waits for a
    // workgroup not yet started would sit out its whole wait at every meeting point. And only for
    // single-output trees, whose root launch is bound by the memory traffic the meetings save; with
    // several outputs the records are found in the L2 anyway (the workgroups of the other outputs
    // asked for them) and the waiting is all that is left (2M x 200, 8 outputs: 1.27 ms with, 0.95 ms without)
    kRoot && a.K == 1 && a.w.n_gk > 1 && a.w.all_resident && a.w.n_chunks <= kPairSyncSlots && a.sync_every > 0 ? hs.pair_sync : nullptr,
    sink);
  return LBT_OK;
}
template <typename BinT, int BV, bool kEmbed>
int launch_binned(hipStream_t stream, const HistSetup& hs, const BinnedArgs& a, const HistBatch& b, unsigned grid,
                  bool root, const PartialSink& sink)
{
  if constexpr (BV == 16) {
    if (a.stripes.log_w >= 0) {
      auto spread = [&](auto per_c) {
        constexpr int kPer = decltype(per_c)::value;
        if (root) return launch_binned_as<BinT, BV, kEmbed, true, true, kPer>(stream, hs, a, b, grid, sink);
        return launch_binned_as<BinT, BV, kEmbed, false, true, kPer>(stream, hs, a, b, grid, sink);
      };
      switch (a.stripes.per) {
        case 12: return spread(std::integral_constant<int, 12>{});
        case 13: return spread(std::integral_constant<int, 13>{});
        case 14: return spread(std::integral_constant<int, 14>{});
        case 16:
          if constexpr (!kEmbed) return spread(std::integral_constant<int, 16>{});
          break;
        default: break;
      }
      if (root) return launch_binned_as<BinT, BV, kEmbed, true, true>(stream, hs, a, b, grid, sink);
      return launch_binned_as<BinT, BV, kEmbed, false, true>(stream, hs, a, b, grid, sink);
    }
  }
  if (root) return launch_binned_as<BinT, BV, kEmbed, true, false>(stream, hs, a, b, grid, sink);
  return launch_binned_as<BinT, BV, kEmbed, false, false>(stream, hs, a, b, grid, sink);
}

// As many resident workgroups as the LDS allows per CU; row-tile ranges come in multiples
// of 8 (one per XCD).
int fill_walk(TileWalk& w, const HistBatch& b, int n_cu, int n_groups, int rpp, int unroll, size_t lds_bytes,
              unsigned* grid)
{
  w.j0          = b.j0;
  w.n_nodes     = b.n_nodes;
  w.level_first = b.level_first;
  w.rpp         = rpp;
  w.tile_rows   = rpp * unroll;
  w.n_gk        = n_groups * b.K;
  const int64_t max_tiles = (b.n_rows + w.tile_rows - 1) / w.tile_rows + b.n_nodes;
  const int per_cu = lds_bytes * 2 <= 160 * 1024 ? 2 : 1;
  int64_t per_xcd  = std::max<int64_t>(1, (per_cu * n_cu / 8) / w.n_gk);
  per_xcd         = std::min<int64_t>(per_xcd, std::max<int64_t>(1, (max_tiles + 7) / 8));
  w.n_chunks      = static_cast<int>(per_xcd * 8);
  *grid           = static_cast<unsigned>(per_xcd * 8 * w.n_gk);
  w.all_resident  = static_cast<int64_t>(*grid) <= static_cast<int64_t>(per_cu) * n_cu;
  return LBT_OK;
}

PlanArgs plan_of(const HistSetup& hs, const HistBatch& b, const TileWalk& w)
{
  PlanArgs p{b.j0, b.j0 + b.n_nodes, b.level_first, b.seg, b.node_sums, b.hist, w.tile_rows, hs.tiles, hs.meta, b.level_total, nullptr,
             hs.binned != nullptr ? hs.partial_count : nullptr, hs.partial_list_count, 0};
  const int64_t max_tiles = (b.n_rows + w.tile_rows - 1) / w.tile_rows + b.n_nodes;
  p.blocks                = static_cast<int>((max_tiles + kPlanThreads - 1) / kPlanThreads);
  return p;
}

// rows per lane and tile on cached bins below the root
int level_unroll(const HistSetup& hs) { return hs.bvec == 16 ? kBinnedUnroll / 2 : kBinnedUnroll; }

template <typename T>
int hist_launch_t(hipStream_t stream, const HistSetup& hs, const HistBatch& b, int depth)
{
  const bool use_cache = hs.binned != nullptr;
  int device = 0, n_cu = 256;
  LBT_HIP(hipGetDevice(&device));
  LBT_HIP(hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, device));
  if (use_cache && b.fill_cache) {
    // fill the bin cache: rows split evenly over as many workgroups as are resident at once
    // X read once, one bin written per value; with embedded gradients also one pair read and
    // one written per row and histogram group
    ProfScope ps(LBT_PROF_BINNING, stream,
                 static_cast<double>(b.n_rows) * b.F * (sizeof(T) + static_cast<double>(hs.bin_bytes)) +
                   (hs.embed ? static_cast<double>(b.n_rows) * 8.0 * (1 + hs.n_groups) : 0.0));
    BinRowsArgs<T> a;
    a.F            = b.F;
    a.n_rows       = b.n_rows;
    a.proposals    = static_cast<const T*>(b.proposals);
    a.row_pointers = b.row_pointers;
    a.bin_feature  = b.bin_feature;
    a.sgroups      = hs.sgroups;
    a.tables       = hs.tables;
    a.map_x        = static_cast<const T*>(hs.map_x);
    a.map_t        = hs.map_t;
    a.straight     = hs.straight;
    a.cells        = hs.cells;
    a.search_steps = hs.search_steps;
    a.n_sgroups    = hs.n_sgroups;
    a.rpp          = hs.rpp;
    a.share        = hs.share;
    a.lanes        = hs.bin_lanes;
    a.rec          = hs.rec;
    const int per_cu = hs.lds_bytes * 2 <= 160 * 1024 ? 2 : 1;
    int64_t per_xcd  = std::max<int64_t>(1, (per_cu * n_cu / 8) / hs.n_sgroups);
    per_xcd          = std::min<int64_t>(per_xcd, std::max<int64_t>(1, (b.n_rows / (hs.rpp * kUnroll) + 7) / 8));
    // the kernel addresses a chunk's rows with 32-bit byte offsets
    const int64_t widest = std::max<int64_t>(static_cast<int64_t>(b.F) * sizeof(T), hs.max_rec_stride);
    while ((b.n_rows / (per_xcd * 8) + 34) * widest >= (int64_t(1) << 31)) per_xcd *= 2;
    a.n_chunks       = static_cast<int>(per_xcd * 8);
    const unsigned grid = static_cast<unsigned>(per_xcd * 8 * hs.n_sgroups);
    int rc = LBT_OK;
    if (hs.vec == 4) {
      rc = launch_bin_rows_t<T, 4>(stream, hs, a, b, grid);
    } else if (hs.vec == 2) {
      rc = launch_bin_rows_t<T, 2>(stream, hs, a, b, grid);
    } else {
      rc = launch_bin_rows_t<T, 1>(stream, hs, a, b, grid);
    }
    LBT_TRY(rc);
  }
  // the root launch on cached bins also writes the feature-major copy (four rows per lane and tile)
  const bool root = use_cache && b.identity && hs.bins_t != nullptr;
  TileWalk w;
  unsigned grid = 0;
  LBT_TRY(fill_walk(w, b, n_cu, hs.n_groups, use_cache ? hs.brpp : hs.rpp,
                    use_cache ? (root ? 4 : level_unroll(hs)) : kUnroll,
                    use_cache ? hs.blds_bytes : hs.lds_bytes, &grid));
  if (!b.planned) {
    ProfScope ps(LBT_PROF_OTHER, stream);
    PlanArgs p = plan_of(hs, b, w);
    if (root && w.n_chunks <= kPairSyncSlots) p.pair_sync = hs.pair_sync;
    if (b.n_nodes <= kPlanFusedNodes) {
      plan_expand_tiles_kernel<<<p.blocks, kPlanThreads, 0, stream>>>(p);
    } else {
      plan_tiles_kernel<<<1, kPlanThreads, 0, stream>>>(b.j0, b.j0 + b.n_nodes, b.level_first, b.seg, b.node_sums, b.hist, w.tile_rows,
                                                        hs.tile_start, hs.meta, b.level_total);
      expand_tiles_kernel<<<p.blocks, kPlanThreads, 0, stream>>>(b.j0, b.n_nodes, b.level_first, b.seg, hs.tile_start, hs.meta,
                                                                 w.tile_rows, hs.tiles, p.pair_sync, p.partial_count,
                                                                 hs.partial_list_count);
    }
  }
  if (use_cache) {
    BinnedArgs a;
    a.w            = w;
    a.rec          = hs.rec;
    a.K            = b.K;
    a.row_pointers = b.row_pointers;
    a.groups       = hs.groups;
    a.hist         = b.hist;
    a.stripes      = Stripes{hs.stripe_log, hs.stripe_bins, hs.spread};
    a.lanes        = hs.even_lanes;
    a.sync_every   = kPairSyncTiles;
    PartialSink sink{hs.partials, hs.partial_lists, hs.partial_list_count, hs.partial_count, 0, hs.partial_stride};
    if (hs.partials != nullptr && static_cast<int64_t>(w.n_nodes) * w.n_gk <= kPartialMaxLists)
      sink.slots = hs.partial_slots;
    {
      ProfScope ps(LBT_PROF_HISTOGRAM, stream, 0.0, depth);
      int rc;
      if (hs.bin_bytes == 1)
        rc = hs.embed ? launch_binned<uint8_t, 16, true>(stream, hs, a, b, grid, root, sink)
                      : launch_binned<uint8_t, 16, false>(stream, hs, a, b, grid, root, sink);
      else
        rc = hs.embed ? launch_binned<uint16_t, 4, true>(stream, hs, a, b, grid, root, sink)
                      : launch_binned<uint16_t, 4, false>(stream, hs, a, b, grid, root, sink);
      LBT_TRY(rc);
    }
    if (sink.slots > 0) {
      // timed with the scan, which is the other pass over the finished histograms
      ProfScope ps(LBT_PROF_SCAN, stream);
      // the stride is the widest group in bins; near the root, where few lists are long, the slots of
      // a list are dealt to several workgroups
      const int lists      = w.n_nodes * w.n_gk;
      const int bin_chunks = (sink.stride + kHistThreads - 1) / kHistThreads;
      const int split      = std::max(1, std::min(16, 256 / (lists * bin_chunks)));
      dim3 rgrid(static_cast<unsigned>(bin_chunks), static_cast<unsigned>(lists), static_cast<unsigned>(split));
      reduce_partials_kernel<<<rgrid, kHistThreads, 0, stream>>>(sink, a.K, w.n_gk / a.K, a.groups, a.row_pointers, a.hist,
                                                                 w.level_first + w.j0, a.stripes);
    }
    return LBT_OK;
  }
  ProfScope ps(LBT_PROF_HISTOGRAM, stream, 0.0, depth);
  HistArgs<T> a;
  a.w            = w;
  a.F            = b.F;
  a.n_rows       = b.n_rows;
  a.K            = b.K;
  a.proposals    = static_cast<const T*>(b.proposals);
  a.row_pointers = b.row_pointers;
  a.groups       = hs.groups;
  a.tables       = hs.tables;
  a.map_x        = static_cast<const T*>(hs.map_x);
  a.map_t        = hs.map_t;
  a.cells        = hs.cells;
  a.search_steps = hs.search_steps;
  a.hist         = b.hist;
  if (hs.vec == 4) {
    if constexpr (sizeof(T) == 4) return launch_search_rows<T, 4>(stream, hs, a, b, grid, b.identity);
  }
  if (hs.vec == 2) return launch_search_rows<T, 2>(stream, hs, a, b, grid, b.identity);
  return launch_search_rows<T, 1>(stream, hs, a, b, grid, b.identity);
}

// Packs consecutive features, `unit` at a time, into groups whose LDS need
// (bytes_of(feature)) stays within the budget and whose rows take at most half a
// workgroup of lanes (lane_vec features per lane; the binning pass has more, see bin_lanes); a second pass balances widths.
// more_groups: that many groups beyond the fewest the budget allows.
template <typename BytesOf>
size_t pack_groups(int F, int unit, int lane_vec, size_t budget, BytesOf bytes_of, std::vector<int32_t>& groups,
                   int more_groups = 0)
{
  const int max_lanes = kHistThreads / 2;  // of features
  size_t lds          = 0;
  auto pack = [&](int target) {
    groups.assign(1, 0);
    lds        = 0;
    size_t cur = 0;
    int width  = 0;
    for (int f = 0; f < F; f += unit) {
      size_t cb = 0;
      for (int i = f; i < std::min(F, f + unit); i++) cb += bytes_of(i);
      if (width > 0 && (cur + cb > budget || width + unit > target || (width + unit + lane_vec - 1) / lane_vec > max_lanes)) {
        groups.push_back(f);
        lds   = std::max(lds, cur);
        cur   = 0;
        width = 0;
      }
      cur += cb;
      width += unit;
    }
    groups.push_back(F);
    lds = std::max(lds, cur);
  };
  pack(F + unit);  // fewest groups the LDS allows
  const int n_min = std::min(static_cast<int>(groups.size()) - 1 + more_groups, (F + unit - 1) / unit);
  int target      = (F + n_min - 1) / n_min;
  target          = ((target + unit - 1) / unit) * unit;
  pack(target);    // same count where the budget allows, balanced widths
  return lds;
}

int rows_per_pass(const std::vector<int32_t>& groups, int vec)
{
  int rpp = kHistThreads;
  for (size_t g = 0; g + 1 < groups.size(); g++) {
    int lanes = (groups[g + 1] - groups[g] + vec - 1) / vec;
    rpp       = std::min(rpp, kHistThreads / lanes);
  }
  return rpp;
}

// Lanes that share a record of the binning pass, where all records have 32 bytes of which 16 hold the bins of one, two or four lanes; more than
// one lane: a single record, whose lanes then are side by side in a wave. 0: not so.
// With lanes of a word each, seven of the eight of a record with four bins search for nothing, and bins written byte by byte are up to 25 stores a row.
// 17,000,000 rows, us with shares and without: floats x 1 225 and 446, x 3 198 and 470, x 4 248 and 391, x 5 226 and 423, x 8 253 and 394, x 9 300
// and 440, x 16 363 and 411; doubles x 1 221 and 457, x 4 288 and 449, x 8 357 and 455, x 16 587 and 599; two-byte bins:
// floats x 3 199 and 467, x 5 226 and 250, doubles x 5 289 and 307.
int share_of_record(const std::vector<int32_t>& groups, const std::vector<RecInfo>& rec, int vec, int bin_bytes)
{
  int share = 1;
  for (size_t g = 0; g < rec.size(); g++) {
    const int lanes = (groups[g + 1] - groups[g] + vec - 1) / vec;
    if (rec[g].size != 32 || lanes * vec * bin_bytes > 16 || lanes > 4 || (lanes > 2 && vec * bin_bytes != 4)) return 0;
    share = std::max(share, lanes <= 2 ? lanes : 4);
  }
  return share > 1 && rec.size() > 1 ? 0 : share;
}

// The lanes that hold a row in the binning pass: two entries for each search group, {where its lanes begin,
// how many} and {bytes between the rows of its plane, where that begins in units of kPlaneAlign}, then the lanes. A lane is
// {first feature, kind + 4 * its first byte in the plane's row} and holds vec * bin_bytes bytes of a record; kind 0: bins, 1: zeros, 2 and 3: the
// words of the gradient pair (2: both, where a lane holds two words). A search group has the lanes of its features and, behind a
// record's last ones, those of the rest of the record. share > 0: a record has that many lanes, of 32 / share bytes each; kind 1: without
// features (share_of_record). Otherwise, where a lane has less than four bytes, there are lanes of bins only {record, ...}, kind 1: a record's last one.
// Returns the rows that a workgroup takes side by side: as many as fit, or up to an eighth fewer that are whole cache lines; 0 where a
// row does not fit. (A search group has up to 512 lanes of features and up to 13 more for each of its records. The LDS holds the proposals
// of 40,000 bins, and a record has 19,000 of them but where more records fill the chip better: seven at the most, some 600 lanes of the 1024.)
int bin_lanes(const std::vector<int32_t>& sgroups, const std::vector<int32_t>& groups, const std::vector<RecInfo>& rec,
              int vec, int bin_bytes, int share, std::vector<int2>& lanes)
{
  const int n_s = static_cast<int>(sgroups.size()) - 1, own = vec * bin_bytes;
  lanes.assign(2 * static_cast<size_t>(n_s), make_int2(0, 0));
  int rpp      = kHistThreads;
  size_t group = 0;
  for (int s = 0; s < n_s; s++) {
    const int begin = static_cast<int>(lanes.size());
    for (int f = sgroups[s]; f < sgroups[s + 1]; f += vec) {
      while (groups[group + 1] <= f) group++;
      const RecInfo& ri = rec[group];
      const int at      = ri.in_row + (f - groups[group]) * bin_bytes;
      const bool last   = f + vec >= groups[group + 1];
      if (share > 0) {
        for (int nth = (f - groups[group]) / vec; nth < share; nth++) {
          const bool own_bins = nth == (f - groups[group]) / vec;
          lanes.push_back(make_int2(f, (own_bins ? 0 : 1) + 4 * (ri.in_row + nth * 32 / share)));
          if (!last) break;
        }
        continue;
      }
      lanes.push_back(make_int2(own >= 4 ? f : static_cast<int>(group), (own < 4 && last ? 1 : 0) + 4 * at));
      if (own < 4 || !last) continue;
      const int end = ri.in_row + ri.size;
      for (int byte = at + own; byte < end; byte += own) {
        const bool pair = ri.q_off >= 0 && byte >= end - 8;
        lanes.push_back(make_int2(f, (pair ? (byte == end - 8 ? 2 : 3) : 1) + 4 * byte));
      }
    }
    const int n      = static_cast<int>(lanes.size()) - begin;
    lanes[2 * s]     = make_int2(begin, n);
    lanes[2 * s + 1] = make_int2(rec[group].stride, static_cast<int>((rec[group].base - rec[group].in_row) / kPlaneAlign));
    rpp              = std::min(rpp, kHistThreads / n);
  }
  auto whole_lines = [&](int rows) {
    for (const RecInfo& ri : rec)
      if (static_cast<int64_t>(rows) * ri.stride % 128 != 0) return false;
    return true;
  };
  for (int fewer = rpp; fewer >= std::max(1, rpp - rpp / 8); fewer--)
    if (whole_lines(fewer)) return fewer;
  return rpp;
}

template <typename BytesOf>
size_t widest_group(const std::vector<int32_t>& groups, BytesOf bytes_of)
{
  size_t need = 0;
  for (size_t g = 0; g + 1 < groups.size(); g++) {
    size_t sb = 0;
    for (int f = groups[g]; f < groups[g + 1]; f++) sb += bytes_of(f);
    need = std::max(need, sb);
  }
  return need;
}

}  // namespace

// The small tables hist_prepare sends to the device (feature groups, record layouts) are carved
// from one block of the workspace that holds nothing else. They are gathered in one pinned
// buffer per host thread and sent with one copy: every separate small copy costs about 10 us of
// the stream's time.
struct Upload {
  struct Item {
    void* dst;
    const void* src;
    size_t bytes;
  };
  std::vector<Item> items;
  void add(void* dst, const void* src, size_t bytes)
  {
    if (bytes > 0) items.push_back({dst, src, bytes});
  }
  // [block, block + block_bytes) is the part of the workspace set aside for these tables: the one
  // copy overwrites all of it (zeros between the tables). Items outside it, or no pinned buffer,
  // and every table travels by itself.
  int send(hipStream_t stream, void* block, size_t block_bytes, SmallTables* small)
  {
    // with the next launch, where they are few
    size_t words = 0;
    bool fits    = items.size() <= SmallTables::kMost;
    for (const Item& it : items) {
      fits = fits && it.bytes % 4 == 0;
      words += it.bytes / 4;
    }
    small->n = small->used = 0;
    if (fits && words <= SmallTables::kWords) {
      for (const Item& it : items) {
        small->to[small->n]    = static_cast<uint32_t*>(it.dst);
        small->at[small->n]    = small->used;
        small->words[small->n] = static_cast<int>(it.bytes / 4);
        std::memcpy(small->data + small->used, it.src, it.bytes);
        small->used += small->words[small->n++];
      }
      items.clear();
    }
    if (items.empty()) return LBT_OK;
    char* const lo = static_cast<char*>(block);
    bool together  = block != nullptr && block_bytes > 0 && block_bytes <= (size_t(1) << 22);
    for (const Item& it : items) {
      const char* d = static_cast<const char*>(it.dst);
      together      = together && d >= lo && d + it.bytes <= lo + block_bytes;
    }
    ThreadResources* here = nullptr;
    LBT_TRY(thread_resources_here(&here));
    ThreadResources& tr = *here;
    if (together) {
      if (tr.stage_free == nullptr) {
        if (hipEventCreateWithFlags(&tr.stage_free, hipEventDisableTiming) != hipSuccess) together = false;
      } else {
        // the buffer may still be the source of an earlier call's copy (on another stream)
        LBT_HIP(hipEventSynchronize(tr.stage_free));
      }
      if (together && tr.stage_bytes < block_bytes) {
        if (tr.stage != nullptr) LBT_HIP(hipHostFree(tr.stage));
        tr.stage       = nullptr;
        tr.stage_bytes = 0;
        if (hipHostMalloc(reinterpret_cast<void**>(&tr.stage), block_bytes + 4096, hipHostMallocDefault) == hipSuccess)
          tr.stage_bytes = block_bytes + 4096;
        else
          together = false;
      }
      if (together) {
        std::memset(tr.stage, 0, block_bytes);
        for (const Item& it : items) std::memcpy(tr.stage + (static_cast<char*>(it.dst) - lo), it.src, it.bytes);
        LBT_HIP(hipMemcpyAsync(lo, tr.stage, block_bytes, hipMemcpyHostToDevice, stream));
        LBT_HIP(hipEventRecord(tr.stage_free, stream));
        items.clear();
        return LBT_OK;
      }
    }
    // pageable sources that the caller reuses: the copies must have read them before this returns
    for (const Item& it : items) LBT_HIP(hipMemcpyAsync(it.dst, it.src, it.bytes, hipMemcpyHostToDevice, stream));
    LBT_HIP(hipStreamSynchronize(stream));
    items.clear();
    return LBT_OK;
  }
};

int hist_prepare(hipStream_t stream, HistSetup& hs, bool is_f64, int F, int K, int64_t n_rows,
                 const std::vector<int32_t>& rp, const void* proposals, const int32_t* row_pointers,
                 const void* X, const RootArgs* root)
{
  const size_t elem = is_f64 ? 8 : 4;
  hs.is_f64         = is_f64;
  hs.n_features     = F;
  // widest aligned vector of features a lane can load from X
  int vec = is_f64 ? 2 : 4;
  while (vec > 1 && (F % vec != 0 || reinterpret_cast<uintptr_t>(X) % 16 != 0)) vec >>= 1;
  // The binning pass keeps the full width for a feature count that is no multiple of it (the
  // last lane of a row then owns fewer features); the kernel that searches X itself does not.
  hs.ragged = false;
  if (hs.binned != nullptr) {
    const int full = F >= 4 ? 4 : std::min(F, 2);
    if (vec < full && reinterpret_cast<uintptr_t>(X) % elem == 0) {
      vec       = full;
      hs.ragged = F % full != 0;
      if (!hs.ragged && reinterpret_cast<uintptr_t>(X) % 16 != 0) hs.ragged = true;  // same loads: element alignment
    }
  }
  hs.vec = vec;
  int max_feature_bins = 1;
  for (int f = 0; f < F; f++) max_feature_bins = std::max(max_feature_bins, rp[f + 1] - rp[f]);
  hs.search_steps = 0;
  while ((1 << hs.search_steps) < max_feature_bins + 1) hs.search_steps++;
  const bool cached = hs.binned != nullptr;
  hs.bin_bytes      = max_feature_bins <= 256 ? 1 : 2;
  // cached bins a lane of the histogram kernel loads at once: 16 one-byte or 4 two-byte bins
  hs.bvec  = !cached ? 1 : (hs.bin_bytes == 1 ? 16 : 4);
  hs.embed = cached && K == 1;

  // LDS a feature needs. Search side: proposals and a lookup table, plus the packed
  // sub-histogram when the same kernel accumulates (cache off). Histogram side with the
  // cache: the packed sub-histogram only.
  auto search_bytes = [&](int f, int cells) {
    return static_cast<size_t>(rp[f + 1] - rp[f]) * (cached ? elem : 8 + elem) +
           static_cast<size_t>(cells) / kCellsPerEntry * sizeof(uint2) +
           (cached ? kProbePad * elem : 0);
  };
  auto hist_bytes = [&](int f) { return static_cast<size_t>(rp[f + 1] - rp[f]) * 8; };

  // search groups: as few as the LDS allows with the smallest table ...
  // host copies of the tables; Upload::send has read them when it returns (it copies them into
  // the thread's pinned buffer, or waits for the copies that read them directly)
  static thread_local std::vector<int32_t> sgroups, groups;
  static thread_local std::vector<RecInfo> rec;
  static thread_local std::vector<int2> lanes;
  const size_t search_budget = kLdsBudget - 128;  // room for the entries in front, the slack entries and alignment
  size_t budget              = search_budget;
  for (;;) {
    pack_groups(F, vec, vec, budget, [&](int f) { return search_bytes(f, 64); }, sgroups);
    const size_t need = widest_group(sgroups, [&](int f) { return search_bytes(f, 64); });
    if (need <= search_budget) break;
    if (budget <= 16 * 1024) {
      set_error("a feature group does not fit the LDS (%zu bytes)", need);
      return LBT_ERR_UNSUPPORTED;
    }
    budget -= 16 * 1024;
  }
  // ... half as many groups again where that buys a table of eight cells per proposal (wide
  // inputs: with 125 features of 256 proposals in a group only two cells per proposal are left,
  // and the search, no longer hidden behind the loads, sets the pace; a further group costs one
  // more partly used cache line per row) ...
  {
    const int n_min   = static_cast<int>(sgroups.size()) - 1;
    const int allowed = n_min + n_min / 2;
    std::vector<int32_t> trial;
    for (int c = kMaxCells; allowed > n_min && c >= 128; c >>= 1) {
      if (c > 8 * std::max(16, max_feature_bins)) continue;
      pack_groups(F, vec, vec, search_budget, [&](int f) { return search_bytes(f, c); }, trial);
      if (widest_group(trial, [&](int f) { return search_bytes(f, c); }) > search_budget) continue;
      if (static_cast<int>(trial.size()) - 1 > allowed) continue;
      sgroups = trial;
      break;
    }
  }
  // ... then the largest table, up to eight cells per proposal, that still fits these groups
  int cells = 64;
  size_t search_lds = widest_group(sgroups, [&](int f) { return search_bytes(f, 64); });
  for (int c = 128; c <= kMaxCells && c <= 8 * std::max(16, max_feature_bins); c <<= 1) {
    const size_t need = widest_group(sgroups, [&](int f) { return search_bytes(f, c); });
    if (need > search_budget) break;
    cells      = c;
    search_lds = need;
  }
  hs.cells     = cells;
  hs.n_sgroups = static_cast<int>(sgroups.size()) - 1;
  hs.lds_bytes = (search_lds + (cached ? (kProbePad + kProbeSlack) * elem : 8) + 15) & ~size_t(15);
  hs.rpp       = rows_per_pass(sgroups, vec);
  Upload up;
  up.add(hs.sgroups, sgroups.data(), sizeof(int32_t) * sgroups.size());

  rec.clear();
  if (!cached) {
    // one kernel searches and accumulates: the search groups are the histogram groups
    groups       = sgroups;
    hs.n_groups  = hs.n_sgroups;
    hs.groups    = hs.sgroups;
  } else {
    // histogram groups hold whole lanes of the binning pass (multiples of vec features)
    const size_t hbudget = kLdsBudget - 8 * kHistThreads;  // one spare slot per lane
    pack_groups(F, vec, hs.bvec, hbudget, hist_bytes, groups);
    {
      // A launch has one workgroup per (row range, group, output) and as many row ranges as keep
      // every CU busy once: 3 groups x 8 outputs are 24 workgroups per row range, of which a
      // 32-CU XCD takes one set and leaves 8 CUs idle. One or two groups more are taken when that
      // fills the chip a quarter better (the atomics per row stay the same, the record requests
      // per row grow with the groups).
      int device = 0, n_cu = 256;
      LBT_HIP(hipGetDevice(&device));
      LBT_HIP(hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, device));
      const int slots = std::max(1, n_cu / 8);  // workgroups of this size that an XCD runs at once
      auto filled = [&](int n_groups) {
        const int n_gk = n_groups * K;
        if (n_gk <= slots) return static_cast<double>(slots / n_gk * n_gk) / slots;
        const int rounds = (n_gk + slots - 1) / slots;
        return static_cast<double>(n_gk) / (static_cast<double>(rounds) * slots);
      };
      const int n0 = static_cast<int>(groups.size()) - 1;
      int best     = 0;
      for (int more = 1; more <= 2; more++)
        if (filled(n0 + more) >= 1.25 * filled(n0) && filled(n0 + more) > filled(n0 + best)) best = more;
      if (best > 0) pack_groups(F, vec, hs.bvec, hbudget, hist_bytes, groups, best);
    }
    // As many groups that lie within one search group each, where that is possible: every search group then has planes of its own in the
    // cache and writes whole cache lines (2,000,000 x 200, search groups of 100: records of 52, 52, 52 and 44 features, of
    // which the second is written by two workgroups, 681 us; 52, 48, 52 and 48 in two planes 483).
    bool planes = hs.n_sgroups == 1;
    if (!planes) {
      const int n_s = hs.n_sgroups, n_all = static_cast<int>(groups.size()) - 1;
      static thread_local std::vector<int32_t> aligned, part;
      for (int more = 0; more <= 2 && !planes; more++) {
        aligned.assign(1, 0);
        for (int g = 0; g < n_s; g++) {
          const int f0 = sgroups[g];
          pack_groups(sgroups[g + 1] - f0, vec, hs.bvec, hbudget, [&](int f) { return hist_bytes(f0 + f); }, part, more);
          for (size_t i = 1; i < part.size(); i++) aligned.push_back(f0 + part[i]);
        }
        const int n = static_cast<int>(aligned.size()) - 1;
        if (n > n_all) break;
        planes = n == n_all;
      }
      if (planes) groups = aligned;
    }
    const size_t blds = widest_group(groups, hist_bytes);
    if (blds > hbudget) {
      set_error("the bins of one feature group do not fit the LDS (%zu bytes)", blds);
      return LBT_ERR_UNSUPPORTED;
    }
    hs.n_groups   = static_cast<int>(groups.size()) - 1;
    hs.blds_bytes = (blds + 8 * kHistThreads + 15) & ~size_t(15);
    hs.partial_stride = static_cast<int>(blds / 8);  // bins of the widest group
    // The striped layout (one-byte bins) takes max bins x W words, W the power of two that holds the
    // widest group: used whenever that fits the LDS with the groups the packed layout would have.
    hs.stripe_log  = -1;
    hs.stripe_bins = 0;
    if (hs.bin_bytes == 1) {
      int widest = 1;
      for (int g = 0; g < hs.n_groups; g++) widest = std::max(widest, groups[g + 1] - groups[g]);
      int log_w = 4;
      while ((1 << log_w) < widest) log_w++;
      const size_t need = static_cast<size_t>(max_feature_bins) * 8 << log_w;
      if ((1 << log_w) <= kStripeMaxW && need <= kLdsBudget - 8 * 1024) {
        hs.stripe_log     = log_w;
        hs.stripe_bins    = max_feature_bins;
        hs.blds_bytes     = (need + 15) & ~size_t(15);
        hs.partial_stride = static_cast<int>(need / 8);
      }
    }
    if (hs.partial_stride > kPartialStrideMax) hs.partials = nullptr;
    hs.brpp       = rows_per_pass(groups, hs.bvec);
    up.add(hs.groups, groups.data(), sizeof(int32_t) * groups.size());
    // record layout of every histogram group
    const int chunk = hs.bvec * hs.bin_bytes;  // bytes a lane of the histogram kernel loads
    // The records of a row lie side by side ([row][group]): the binning pass, whose lanes hold a
    // whole row, then writes one contiguous piece per row, and the workgroups that read the
    // groups of the same rows at the same time share the cache lines.
    rec.resize(hs.n_groups);
    int pitch          = 0;  // of the rows of a plane; without planes of the whole cache
    int widest_pitch   = 0;
    int64_t plane_base = 0;
    hs.row_bytes       = 0;
    auto end_plane     = [&](int from, int to) {
      for (int g = from; g < to; g++) rec[g].stride = pitch;
      widest_pitch = std::max(widest_pitch, pitch);
      hs.row_bytes += pitch;
      plane_base   = (plane_base + n_rows * static_cast<int64_t>(pitch) + kPlaneAlign - 1) / kPlaneAlign * kPlaneAlign;
      pitch        = 0;
    };
    int plane_first = 0, sgroup = 0;
    for (int g = 0; g < hs.n_groups; g++) {
      if (planes && groups[g] >= sgroups[sgroup + 1]) {
        end_plane(plane_first, g);
        plane_first = g;
        sgroup++;
      }
      const int gs        = groups[g + 1] - groups[g];
      const int bins_end  = gs * hs.bin_bytes;
      const int chunk_end = (bins_end + chunk - 1) / chunk * chunk;
      RecInfo& ri         = rec[g];
      ri.bins_end         = bins_end;
      // bins, zeros up to the end of the record, the gradient pair (if embedded) in the last 8
      // bytes: every byte of a record is written, so no cache line reaches memory in parts
      const int used = std::max(chunk_end, hs.embed ? (bins_end + 7) / 8 * 8 + 8 : 0);
      ri.size        = (used + 31) / 32 * 32;
      ri.q_off       = hs.embed ? ri.size - 8 : -1;
      ri.zero_end    = hs.embed ? ri.q_off : ri.size;
      ri.base        = plane_base + pitch;
      ri.in_row      = pitch;
      pitch += ri.size;
    }
    end_plane(plane_first, hs.n_groups);
    hs.max_rec_stride = widest_pitch;
    hs.max_bins       = max_feature_bins;
    hs.pieces         = 0;
    for (int g = 0; g < hs.n_groups; g++) hs.pieces += (rec[g].bins_end + 15) / 16;
    // the same lanes per row for all groups (see binned_histogram_kernel): when the striped layout is
    // used, the records carry the gradient pair (one output: the groups' workgroups are bound by the
    // memory traffic they can share) and every record is long enough for the widest group's lanes
    hs.even_lanes = 0;
    if (hs.stripe_log >= 0 && hs.embed && hs.n_groups > 1) {
      int lanes = 0;
      for (int g = 0; g < hs.n_groups; g++) lanes = std::max(lanes, (groups[g + 1] - groups[g] + hs.bvec - 1) / hs.bvec);
      bool fits = true;
      for (int g = 0; g < hs.n_groups; g++) fits = fits && lanes * chunk <= rec[g].size;
      fits = fits && lanes * hs.bvec <= (1 << hs.stripe_log);
      if (fits) hs.even_lanes = lanes;
    }
    // Four lanes per row that share its bins evenly (kPer of binned_histogram_kernel), where the widest group needs three or
    // four lanes of 16 and all records have the bytes of four; with one output the pair in the last 8 of 64. Groups of up to 48
    // features take four lanes of 12 for three of 16. With few bins the second half of the array, 64 KB behind the first, leaves one
    // workgroup to a CU where two had room, and it pays all the more: trees of depth 8 on 5,000,000 x 50 with 64, 128 and 256 samples
    // 1856, 2065 and 1784 us without, 1611, 1679 and 1774 with it; 600,000 x 50 with 8 outputs 1142, 1305 and 1430, 1016, 1164 and 1394.
    hs.spread = 0;
    if (hs.stripe_log == 6) {
      int widest  = 0;
      bool whole = true;
      for (int g = 0; g < hs.n_groups; g++) {
        widest = std::max(widest, groups[g + 1] - groups[g]);
        whole  = whole && (hs.embed ? rec[g].size == 64 && rec[g].q_off == 56 : rec[g].size >= 64);
      }
      if (whole) {
        hs.spread     = widest <= 48 ? 12 : (widest <= 52 ? 13 : (widest <= 56 ? 14 : 16));
        hs.even_lanes = 4;
        hs.brpp       = kHistThreads / 4;
        hs.blds_bytes = spread_hist_bytes(hs.stripe_bins) + kSpreadMore;
      }
    }
    const int64_t at = plane_base;
    if (static_cast<size_t>(at) > hs.binned_capacity) {
      set_error("bin cache of %lld bytes exceeds the workspace share", static_cast<long long>(at));
      return LBT_ERR_WORKSPACE;
    }
    up.add(hs.rec, rec.data(), sizeof(RecInfo) * rec.size());
    hs.share = share_of_record(groups, rec, vec, hs.bin_bytes);
    hs.rpp   = bin_lanes(sgroups, groups, rec, vec, hs.bin_bytes, hs.share, lanes);
    if (hs.rpp < 1 || lanes.size() > bin_lanes_max(F)) {
      set_error("a row takes %zu lanes of the binning pass", lanes.size());
      return LBT_ERR_INVALID;
    }
    up.add(hs.bin_lanes, lanes.data(), sizeof(int2) * lanes.size());
  }
  SmallTables small{};
  LBT_TRY(up.send(stream, hs.upload_block, hs.upload_bytes, &small));
  ProfScope ps(LBT_PROF_PROPOSALS, stream);
  const RootArgs begin    = root != nullptr ? *root : RootArgs{};
  const int64_t clears    = (begin.n16 + 256 * kClearUnits - 1) / (256 * kClearUnits);
  const unsigned grid     = static_cast<unsigned>(F + 1 + clears);
  if (is_f64)
    build_cells_kernel<double><<<grid, 256, 0, stream>>>(static_cast<const double*>(proposals), row_pointers, F, cells, hs.tables,
                                                         static_cast<double*>(hs.map_x), hs.map_t, hs.straight, small, begin);
  else
    build_cells_kernel<float><<<grid, 256, 0, stream>>>(static_cast<const float*>(proposals), row_pointers, F, cells, hs.tables,
                                                        static_cast<float*>(hs.map_x), hs.map_t, hs.straight, small, begin);
  return LBT_OK;
}

int hist_plan(const HistSetup& hs, const HistBatch& b, PlanArgs* plan)
{
  *plan = PlanArgs{};
  if (hs.binned == nullptr || b.identity || b.fill_cache || b.n_nodes > kPlanFusedNodes) return LBT_OK;
  TileWalk w;
  unsigned grid = 0;
  LBT_TRY(fill_walk(w, b, 256, hs.n_groups, hs.brpp, level_unroll(hs), hs.blds_bytes, &grid));
  *plan = plan_of(hs, b, w);
  return LBT_OK;
}

int hist_launch(hipStream_t stream, const HistSetup& hs, const HistBatch& b, int depth)
{
  if (hs.is_f64) return hist_launch_t<double>(stream, hs, b, depth);
  return hist_launch_t<float>(stream, hs, b, depth);
}

}  // namespace lbt
