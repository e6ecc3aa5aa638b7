// Bookkeeping of the bipartite K/V merge (merging/merge.py:85-232): which
// tokens are destinations, the order in which sources are merged, and every
// output slot's token list.
//
// gpa_merge_order: mask and order of the tokens.  Whether a token is a
// destination follows from its position and its window's drawn cell alone, and
// every frame past the first has the same number of destinations, so a
// token's rank within its class needs only a scan over its own frame: one
// workgroup per frame, no sort and no scatter.
//
// gpa_merge_plan: from the row maxima and their destinations,
//   edge    = source rows by descending maximum, ties by increasing row
//   slots   = [sources past the first r of `edge`, in that order | destinations]
//   lists   = per slot its own token, then the sources merged into it by
//             increasing position (CSR offsets and tokens), and its size.
// Both orders are stable sorts with 32-bit keys: the maxima's bits in
// descending order, and the merged rows' destinations (rows come in increasing
// position, so stability gives the order within a slot, and a slot of any
// length costs the same).
//
// What bounds it: launches and latency, not bytes (137,400 tokens are 2 MB).
// As torch operations this took over 60 launches per merge, three of them
// merge sorts of up to 16 launches.  Here, one of two ways (by_rank below):
//   * Few rows: by counting.  A row's rank is the number of rows before it; the
//     compares are spread over the whole chip, one launch for each order.  A
//     slot's list starts at its own index plus the counted number of merged
//     rows with a smaller destination.
//   * More: least significant digit radix sorts of 8-bit digits (four passes
//     for the maxima, as many for the destinations as their count has bytes).
//     Each pass is two launches over kTile-row blocks (counts per block, then
//     a scatter in which every block sums the counts of the blocks before it;
//     that sum is ~50 rows of 1 KB at 200 frames, cheaper than a third
//     launch), and a slot's start is a binary search in the sorted keys.
// Measured, a whole merge with its K and V against the torch operations: 521
// -> 121 us at 4 frames (70 -> 9 launches, the plan's two 6 us each), 1,394 ->
// 1,085 us at 100 frames (83 -> 21 launches; the order 5.5 us, the plan ~115 us
// of the GPU's time).
#include "gpa_common.h"

namespace gpa {
namespace {

constexpr int kDigits = 256;

// ---------------------------------------------------------------------------
// mask and order
// ---------------------------------------------------------------------------

struct OrderArgs {
  const int64_t* cell;   // [frames-1][hsy][wsx], null if no patch is drawn
  int64_t* mask;         // [frames * tpi]: -1 destination, 0 source
  int64_t* order;        // [frames * tpi]: destinations first, each by position
  int64_t tpi, num_dst, per_frame;   // per_frame: destinations of a frame past the first
  int frames, ns, sx, sy, hsy, wsx;
};

constexpr int kOrderThreads = 512;

__global__ __launch_bounds__(kOrderThreads) void merge_order_kernel(OrderArgs a) {
  __shared__ int wave_dst[kOrderThreads / 64];
  const int f = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t start = (int64_t)f * a.tpi;
  int64_t dst = f == 0 ? 0 : a.tpi + (f - 1) * a.per_frame;        // destinations before
  const int64_t row_len = (int64_t)a.wsx * a.sx, drawn = a.cell ? (int64_t)a.hsy * a.sy * row_len : 0;
  for (int64_t p0 = 0; p0 < a.tpi; p0 += kOrderThreads) {
    const int64_t p = p0 + tid, j = p - a.ns;
    bool is_dst = f == 0 || j < 0;
    if (!is_dst && j < drawn) {
      const int64_t y = j / row_len, x = j % row_len;
      const int64_t win = ((int64_t)(f - 1) * a.hsy + y / a.sy) * a.wsx + x / a.sx;
      // A cell outside its window counts as the nearest one inside: every window
      // then has its one destination, and the ranks stay inside `order`.
      const int64_t drawn_cell = a.cell[win], last = (int64_t)a.sy * a.sx - 1;
      is_dst = (drawn_cell < 0 ? 0 : drawn_cell > last ? last : drawn_cell) ==
               (y % a.sy) * a.sx + x % a.sx;
    }
    is_dst = is_dst && p < a.tpi;
    const uint64_t votes = __builtin_amdgcn_ballot_w64(is_dst);
    if (lane == 0) wave_dst[wave] = __builtin_popcountll(votes);
    __syncthreads();
    int before = __builtin_popcountll(votes & ((1ull << lane) - 1)), all = 0;
#pragma unroll
    for (int w = 0; w < kOrderThreads / 64; ++w) {
      if (w < wave) before += wave_dst[w];
      all += wave_dst[w];
    }
    if (p < a.tpi) {
      const int64_t rank = dst + before, n = start + p;
      a.mask[n] = is_dst ? -1 : 0;
      a.order[is_dst ? rank : a.num_dst + (n - rank)] = n;
    }
    dst += all;
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// plan
// ---------------------------------------------------------------------------

struct PlanArgs {
  const void* node_max;      // [B][ns]
  const int64_t* node_idx;   // [B][ns]
  const int64_t* order;      // [N]: num_dst destinations, then ns sources
  int64_t* edge;             // [B][ns]
  int64_t* dst_slot;         // [B][r]
  int64_t* unm_abs;          // [B][ns - r]
  int64_t* src_abs;          // [B][r]
  float* size;               // [B][slots]
  int64_t* offsets;          // [B*slots + 1]
  int64_t* tokens;           // [B][N]
  uint32_t *keys0, *keys1, *vals0, *vals1, *counts;   // scratch of the multi-block path
  int64_t B, N;
  int ns, num_dst, r, passes;   // passes: 8-bit digits of a destination key (0 .. num_dst)
  int blocks;                   // kTile-row blocks of one batch element
};

// Ascending unsigned order of this key is descending order of the value as
// torch sorts it: NaN first, -0 equal to +0.
template <typename T>
__device__ __forceinline__ uint32_t max_key(const void* node_max, int64_t i) {
  const float x = (float)static_cast<const T*>(node_max)[i];
  if (x != x) return 0u;
  const uint32_t u = __float_as_uint(x + 0.0f);
  return ~((u & 0x80000000u) ? ~u : (u | 0x80000000u));
}

// A row's destination as a sort key; an index outside the destinations (no
// score of the row was a number) counts as the nearest one, so that the lists
// stay inside their arrays.
__device__ __forceinline__ uint32_t dst_key(int64_t idx, int num_dst) {
  return (uint32_t)(idx < 0 ? 0 : idx >= num_dst ? num_dst - 1 : idx);
}

// One row of the descending order: rank i holds source row e.  Returns the
// row's key for the second sort: its destination, or num_dst if it is kept.
__device__ __forceinline__ uint32_t place_rank(const PlanArgs& a, int64_t b, int i, uint32_t e) {
  const int unm = a.ns - a.r;
  const int64_t pos = a.order[a.num_dst + e];
  a.edge[b * a.ns + i] = e;
  if (i < a.r) {
    const int64_t idx = a.node_idx[b * a.ns + e];
    a.dst_slot[b * a.r + i] = idx;
    a.src_abs[b * a.r + i] = pos;
    return dst_key(idx, a.num_dst);
  }
  const int s = i - a.r;
  const int64_t slot = b * (unm + a.num_dst) + s;
  a.unm_abs[b * unm + s] = pos;
  a.size[slot] = 1.0f;
  a.offsets[slot] = b * a.N + s;
  a.tokens[b * a.N + s] = pos;
  return (uint32_t)a.num_dst;
}

__device__ __forceinline__ int lower_bound(const uint32_t* keys, int n, uint32_t x) {
  int lo = 0;
  while (n > 0) {
    const int half = n >> 1;
    const bool right = keys[lo + half] < x;
    lo = right ? lo + half + 1 : lo;
    n = right ? n - half - 1 : half;
  }
  return lo;
}

// Destination slot j's list head, offset and size: lo merged rows have a
// smaller destination, up one no larger.
__device__ __forceinline__ void place_dst(const PlanArgs& a, int64_t b, int j, int lo, int up) {
  const int unm = a.ns - a.r;
  const int64_t slot = b * (unm + a.num_dst) + unm + j, off = b * a.N + unm + j + lo;
  a.size[slot] = (float)(1 + up - lo);
  a.offsets[slot] = off;
  a.tokens[off] = a.order[j];
}

// The i-th merged row by (destination, position) in its slot's list.
__device__ __forceinline__ void place_member(const PlanArgs& a, int64_t b, int i, uint32_t key,
                                             uint32_t e) {
  a.tokens[b * a.N + (a.ns - a.r) + (int64_t)key + 1 + i] = a.order[a.num_dst + e];
}

// Ranks of a wave's items among its items of the same digit, in item order
// (item u of all lanes before item u + 1), and the digit counts of the wave
// in cnt (zeroed by the wave).  `live` marks the items that exist.
template <int ITEMS>
__device__ __forceinline__ void wave_rank(const uint32_t (&digit)[ITEMS], const bool (&live)[ITEMS],
                                          uint32_t* cnt, uint32_t (&rank)[ITEMS]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 0; d < kDigits; d += 64) cnt[d + lane] = 0;
  asm volatile("" ::: "memory");
#pragma unroll
  for (int u = 0; u < ITEMS; ++u) {
    uint64_t peers = __builtin_amdgcn_ballot_w64(live[u]);
#pragma unroll
    for (int bit = 0; bit < 8; ++bit) {
      const uint64_t set = __builtin_amdgcn_ballot_w64((digit[u] >> bit) & 1);
      peers &= ((digit[u] >> bit) & 1) ? set : ~set;
    }
    const uint32_t before = __builtin_popcountll(peers & ((1ull << lane) - 1));
    // A wave's LDS operations run in order; the empty asm keeps the
    // compiler from moving the read past the write.
    const uint32_t old = live[u] ? cnt[digit[u]] : 0;
    asm volatile("" ::: "memory");
    if (live[u] && before == 0) cnt[digit[u]] = old + (uint32_t)__builtin_popcountll(peers);
    asm volatile("" ::: "memory");
    rank[u] = old + before;
  }
}

// Exclusive scan of one value per digit (threads 0 .. 255; the others pass
// through the barriers).  part: 4 words of LDS.
__device__ __forceinline__ uint32_t scan_digits(uint32_t x, uint32_t* part) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t sum = x;
#pragma unroll
  for (int w = 1; w < 64; w <<= 1) {
    const uint32_t up = __shfl_up(sum, w);
    if (lane >= w) sum += up;
  }
  if (wave < 4 && lane == 63) part[wave] = sum;
  __syncthreads();
  uint32_t base = 0;
#pragma unroll
  for (int w = 0; w < 3; ++w)
    if (w < wave) base += part[w];
  return base + sum - x;
}

// Ranks by counting.  A workgroup takes 16 rows (or destinations): thread
// (part, row) compares its row with every 16th group of four keys, staged in
// LDS kRankKeys at a time, and the 16 parts' counts meet in LDS.  Keys past
// the end are larger than any that is compared with them.
constexpr int kRankRows = 16, kRankParts = 16, kRankThreads = kRankRows * kRankParts;
constexpr int kRankKeys = 4096;
// Where the two ways cross.  Counting costs a compare per pair of source rows,
// half of one per pair of destination and source row, and ~1 ns per workgroup
// (16 rows or destinations); the radix passes hardly more than their launches.
// Microseconds, counting and radix passes (sources, destinations):
//   B = 1   7,280, 3,677: 26, 82    15,600, 6,309: 82, 88    18,000, 1,400: 95, 87
//   B = 2   9,360, 4,335: 63, 88    11,440, 4,993: 87, 88    13,520, 5,651: 116, 90
//   B = 4   5,200, 3,019: 46, 85    7,280, 3,677: 71, 86     9,360, 4,335: 112, 88
//   B = 16  2,080, 2,032: 34, 65    3,120, 2,361: 58, 73     4,160, 2,690: 100, 86
//   B = 32  1,040, 1,703: 27, 60    2,080, 2,032: 60, 67     3,120, 2,361: 106, 75
//   B = 128, 1,040, 1,703: 85, 66;  B = 300, 64, 20,000: 359, 98
constexpr double kRankWork = 3.1e8;
bool by_rank(int64_t B, int64_t ns, int64_t num_dst) {
  const double n = (double)ns, d = (double)num_dst;
  return ns == 0 || (double)B * (n * (n + d / 2) + 250.0 * (2 * n + d)) <= kRankWork;
}

// The sum over the parts of each row's counts, for the threads of part 0.
__device__ __forceinline__ int sum_parts(int x, int (&part)[kRankParts][kRankRows + 1]) {
  const int r = threadIdx.x % kRankRows;
  __syncthreads();
  part[threadIdx.x / kRankRows][r] = x;
  __syncthreads();
  int sum = 0;
#pragma unroll
  for (int p = 0; p < kRankParts; ++p) sum += part[p][r];
  return sum;
}

// Keys base .. base + n of `key` into LDS, the last group of four filled up;
// all loads first (one at a time, their latency was most of the kernel).
template <typename Key>
__device__ __forceinline__ void stage_keys(Key key, int base, int n, uint32_t (&keys)[kRankKeys]) {
  constexpr int kLoads = kRankKeys / kRankThreads;
  uint32_t k[kLoads];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kLoads; ++u) {
    const int t = u * kRankThreads + threadIdx.x;
    k[u] = key(base + min(t, n - 1));
  }
#pragma unroll
  for (int u = 0; u < kLoads; ++u) {
    const int t = u * kRankThreads + threadIdx.x;
    keys[t] = t < n ? k[u] : 0xffffffffu;
  }
  __syncthreads();
}

// Rows before row i = i0 + r in the order of (key, row), over all parts; key(j)
// gives row j's key, mine is row i's.
template <typename Key>
__device__ __forceinline__ int rank_of(Key key, int ns, int i0, uint32_t mine,
                                       uint32_t (&keys)[kRankKeys],
                                       int (&part)[kRankParts][kRankRows + 1]) {
  const int tid = threadIdx.x, r = tid % kRankRows, p = tid / kRankRows;
  int before = 0;
  for (int base = 0; base < ns; base += kRankKeys) {
    const int n = min(kRankKeys, ns - base), n4 = (n + 3) / 4;
    stage_keys(key, base, n, keys);
#pragma unroll 4
    for (int g = p; g < n4; g += kRankParts) {
      const u32x4 k = *reinterpret_cast<const u32x4*>(&keys[4 * g]);
      const int j = base + 4 * g;
      // A tie goes to the earlier row; the workgroup's own rows come below.
      const uint32_t bound = j < i0 ? mine + 1 : j < i0 + kRankRows ? 0u : mine;
      before += (k[0] < bound) + (k[1] < bound) + (k[2] < bound) + (k[3] < bound);
    }
  }
  if (i0 + p < ns) before += key(i0 + p) < mine + (p < r ? 1u : 0u);
  return sum_parts(before, part);
}

template <typename T>
__global__ __launch_bounds__(kRankThreads) void rank_rows_kernel(PlanArgs a) {
  __shared__ __attribute__((aligned(16))) uint32_t keys[kRankKeys];
  __shared__ int part[kRankParts][kRankRows + 1];
  const int64_t b = blockIdx.y;
  const int i0 = blockIdx.x * kRankRows, i = i0 + threadIdx.x % kRankRows;
  auto key = [&](int j) { return max_key<T>(a.node_max, b * a.ns + j); };
  const int rank = rank_of(key, a.ns, i0, i < a.ns ? key(i) : 0u, keys, part);
  if (threadIdx.x < kRankRows && i < a.ns) a.keys0[b * a.ns + i] = place_rank(a, b, rank, i);
}

__global__ __launch_bounds__(kRankThreads) void rank_lists_kernel(PlanArgs a, int row_blocks) {
  __shared__ __attribute__((aligned(16))) uint32_t keys[kRankKeys];
  __shared__ int part[kRankParts][kRankRows + 1];
  const int64_t b = blockIdx.y;
  const int tid = threadIdx.x, r = tid % kRankRows, p = tid / kRankRows;
  const uint32_t* const in = a.keys0 + b * a.ns;
  if ((int)blockIdx.x < row_blocks) {          // source rows
    const int i0 = blockIdx.x * kRankRows, i = i0 + r;
    const uint32_t mine = i < a.ns ? in[i] : 0u;
    const int rank = rank_of([&](int j) { return in[j]; }, a.ns, i0, mine, keys, part);
    if (p == 0 && i < a.ns && mine < (uint32_t)a.num_dst) place_member(a, b, rank, mine, i);
    return;
  }
  const int j = (blockIdx.x - row_blocks) * kRankRows + r;    // destinations
  int less = 0, upto = 0;
  for (int base = 0; base < a.ns; base += kRankKeys) {
    const int n = min(kRankKeys, a.ns - base), n4 = (n + 3) / 4;
    stage_keys([&](int j) { return in[j]; }, base, n, keys);
#pragma unroll 4
    for (int g = p; g < n4; g += kRankParts) {
      const u32x4 k = *reinterpret_cast<const u32x4*>(&keys[4 * g]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        less += k[e] < (uint32_t)j;
        upto += k[e] <= (uint32_t)j;
      }
    }
  }
  less = sum_parts(less, part);
  upto = sum_parts(upto, part);
  if (p == 0 && j < a.num_dst) place_dst(a, b, j, less, upto);
  if (blockIdx.x == gridDim.x - 1 && b == a.B - 1 && tid == 0)
    a.offsets[a.B * (int64_t)(a.ns - a.r + a.num_dst)] = a.B * a.N;
}

// More rows: kTile rows per block, grid (blocks, B).
constexpr int kSortThreads = 512, kSortItems = 8, kTile = kSortThreads * kSortItems;

// counts[b][block][digit] of the pass at `shift`.  FIRST: the keys come from
// the row maxima (element type T), else from `in`.
template <typename T, bool FIRST>
__global__ __launch_bounds__(kSortThreads) void sort_count_kernel(PlanArgs a, const uint32_t* in,
                                                                  int shift) {
  __shared__ uint32_t hist[kDigits];
  const int tid = threadIdx.x;
  const int64_t b = blockIdx.y;
  if (tid < kDigits) hist[tid] = 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kSortItems; ++u) {
    const int i = blockIdx.x * kTile + u * kSortThreads + tid;
    if (i < a.ns) {
      const uint32_t k = FIRST ? max_key<T>(a.node_max, b * a.ns + i) : in[b * a.ns + i];
      atomicAdd(&hist[(k >> shift) & (kDigits - 1)], 1u);
    }
  }
  __syncthreads();
  if (tid < kDigits) a.counts[(b * a.blocks + blockIdx.x) * kDigits + tid] = hist[tid];
}

// The pass's stable scatter.  FIRST as above; IOTA: the values are the rows.
template <typename T, bool FIRST, bool IOTA>
__global__ __launch_bounds__(kSortThreads) void sort_scatter_kernel(PlanArgs a, const uint32_t* kin,
                                                                    const uint32_t* vin, uint32_t* kout,
                                                                    uint32_t* vout, int shift) {
  constexpr int kW = kSortThreads / 64;
  __shared__ uint32_t cnt[kW][kDigits];
  __shared__ uint32_t sums[2][2][kDigits];     // [half][before this block | all][digit]
  __shared__ uint32_t base[kDigits], part[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t b = blockIdx.y;
  uint32_t k[kSortItems], v[kSortItems], digit[kSortItems], rank[kSortItems];
  bool live[kSortItems];
#pragma unroll
  for (int u = 0; u < kSortItems; ++u) {
    const int i = blockIdx.x * kTile + (wave * kSortItems + u) * 64 + lane;
    live[u] = i < a.ns;
    const int64_t at = b * a.ns + (live[u] ? i : 0);
    k[u] = FIRST ? max_key<T>(a.node_max, at) : kin[at];
    v[u] = IOTA ? (uint32_t)i : vin[at];
    digit[u] = (k[u] >> shift) & (kDigits - 1);
  }
  {
    // Each half of the threads sums every second block's counts of a digit.
    const int d = tid & (kDigits - 1), half = tid >> 8;
    const uint32_t* c = a.counts + b * a.blocks * kDigits + d;
    uint32_t before = 0, all = 0;
#pragma unroll 8
    for (int t = half; t < a.blocks; t += 2) {
      const uint32_t x = c[(int64_t)t * kDigits];
      all += x;
      before += t < (int)blockIdx.x ? x : 0;
    }
    sums[half][0][d] = before;
    sums[half][1][d] = all;
  }
  wave_rank<kSortItems>(digit, live, cnt[wave], rank);
  __syncthreads();
  uint32_t all = 0;
  if (tid < kDigits) {
    uint32_t run = 0;
#pragma unroll
    for (int w = 0; w < kW; ++w) {
      const uint32_t c = cnt[w][tid];
      cnt[w][tid] = run;
      run += c;
    }
    all = sums[0][1][tid] + sums[1][1][tid];
  }
  const uint32_t first = scan_digits(all, part);
  if (tid < kDigits) base[tid] = first + sums[0][0][tid] + sums[1][0][tid];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kSortItems; ++u)
    if (live[u]) {
      const int64_t to = b * a.ns + base[digit[u]] + cnt[wave][digit[u]] + rank[u];
      kout[to] = k[u];
      vout[to] = v[u];
    }
}

constexpr int kPlaceThreads = 256;

__global__ __launch_bounds__(kPlaceThreads) void plan_rank_kernel(PlanArgs a, const uint32_t* rows,
                                                                  uint32_t* keys) {
  const int64_t b = blockIdx.y;
  const int i = blockIdx.x * kPlaceThreads + threadIdx.x;
  if (i >= a.ns) return;
  const uint32_t e = rows[b * a.ns + i];
  keys[b * a.ns + e] = place_rank(a, b, i, e);
}

__global__ __launch_bounds__(kPlaceThreads) void plan_lists_kernel(PlanArgs a, const uint32_t* keys,
                                                                   const uint32_t* rows) {
  const int64_t b = blockIdx.y;
  const int i = blockIdx.x * kPlaceThreads + threadIdx.x;
  if (i < a.num_dst) {
    const uint32_t* k = keys + b * a.ns;
    const int lo = lower_bound(k, a.r, i);
    place_dst(a, b, i, lo, lo + lower_bound(k + lo, a.r - lo, i + 1));
  }
  if (i < a.r) place_member(a, b, i, keys[b * a.ns + i], rows[b * a.ns + i]);
  if (i == 0 && b == a.B - 1) a.offsets[a.B * (int64_t)(a.ns - a.r + a.num_dst)] = a.B * a.N;
}

size_t rank_ws_bytes(int64_t B, int64_t ns) { return (size_t)B * ns * sizeof(uint32_t); }
size_t radix_ws_bytes(int64_t B, int64_t ns) {
  return (size_t)B * (4 * ns + (ns + kTile - 1) / kTile * kDigits) * sizeof(uint32_t);
}

template <typename T>
void plan_launch(const PlanArgs& a, bool rank, hipStream_t s) {
  if (rank) {
    const int row_blocks = (a.ns + kRankRows - 1) / kRankRows;
    const int dst_blocks = (a.num_dst + kRankRows - 1) / kRankRows;
    if (a.ns > 0)
      hipLaunchKernelGGL(rank_rows_kernel<T>, dim3((unsigned)row_blocks, (unsigned)a.B),
                         dim3(kRankThreads), 0, s, a);
    // At least one destination block: the last one closes the offsets.
    hipLaunchKernelGGL(rank_lists_kernel,
                       dim3((unsigned)(row_blocks + (dst_blocks > 0 ? dst_blocks : 1)), (unsigned)a.B),
                       dim3(kRankThreads), 0, s, a, row_blocks);
    return;
  }
  const dim3 grid((unsigned)a.blocks, (unsigned)a.B), block(kSortThreads);
  uint32_t *ki = a.keys0, *vi = a.vals0, *ko = a.keys1, *vo = a.vals1;
  auto swap = [&]() {
    uint32_t* t = ki;
    ki = ko;
    ko = t;
    t = vi;
    vi = vo;
    vo = t;
  };
  hipLaunchKernelGGL((sort_count_kernel<T, true>), grid, block, 0, s, a, ki, 0);
  hipLaunchKernelGGL((sort_scatter_kernel<T, true, true>), grid, block, 0, s, a, ki, vi, ko, vo, 0);
  swap();
  for (int p = 1; p < 4; ++p) {
    hipLaunchKernelGGL((sort_count_kernel<T, false>), grid, block, 0, s, a, ki, 8 * p);
    hipLaunchKernelGGL((sort_scatter_kernel<T, false, false>), grid, block, 0, s, a, ki, vi, ko, vo,
                       8 * p);
    swap();
  }
  const dim3 pblock(kPlaceThreads);
  hipLaunchKernelGGL(plan_rank_kernel, dim3((unsigned)((a.ns + kPlaceThreads - 1) / kPlaceThreads), (unsigned)a.B),
                     pblock, 0, s, a, vi, ko);
  swap();      // the new keys; their values are the rows themselves
  for (int p = 0; p < a.passes; ++p) {
    hipLaunchKernelGGL((sort_count_kernel<T, false>), grid, block, 0, s, a, ki, 8 * p);
    if (p == 0)
      hipLaunchKernelGGL((sort_scatter_kernel<T, false, true>), grid, block, 0, s, a, ki, vi, ko, vo, 0);
    else
      hipLaunchKernelGGL((sort_scatter_kernel<T, false, false>), grid, block, 0, s, a, ki, vi, ko, vo,
                         8 * p);
    swap();
  }
  const int most = a.num_dst > a.r ? a.num_dst : a.r;
  hipLaunchKernelGGL(plan_lists_kernel, dim3((unsigned)((most + kPlaceThreads - 1) / kPlaceThreads), (unsigned)a.B),
                     pblock, 0, s, a, ki, vi);
}

}  // namespace
}  // namespace gpa

using namespace gpa;

extern "C" int gpa_merge_order(const int64_t* cell, int64_t frames, int64_t w, int64_t h, int64_t sx,
                               int64_t sy, int64_t num_special, int64_t* mask, int64_t* order,
                               void* stream) {
  gpa_clear_error();
  // Without a cell no window is looked at, and of one frame every token is a
  // destination: only the sizes that are used have to make sense.
  const int64_t most = 0x7fffffff;
  if (frames < 0 || (frames > 1 && num_special < 0) ||
      (cell && (w < 0 || h < 0 || sx <= 0 || sy <= 0))) {
    gpa_set_error("gpa_merge_order: negative size or empty window");
    return GPA_E_INVALID;
  }
  const bool fits = frames <= most && w <= most && w >= -most && h <= most && h >= -most &&
                    num_special <= most && num_special >= -most && (!cell || (sx <= most && sy <= most));
  const int64_t tpi = fits ? w * h + num_special : 0;
  if (!fits || tpi > most) {
    gpa_set_error("gpa_merge_order: %lld frames of %lld x %lld patches exceed the grid limit",
                  (long long)frames, (long long)w, (long long)h);
    return GPA_E_UNSUPPORTED;
  }
  if (tpi < 0) {
    gpa_set_error("gpa_merge_order: negative frame size");
    return GPA_E_INVALID;
  }
  if (frames == 0 || tpi == 0) return GPA_OK;
  if (!mask || !order) {
    gpa_set_error("gpa_merge_order: null pointer");
    return GPA_E_INVALID;
  }
  OrderArgs a{};
  a.hsy = cell ? (int)(h / sy) : 0;
  a.wsx = cell ? (int)(w / sx) : 0;
  a.cell = a.hsy > 0 && a.wsx > 0 ? cell : nullptr;
  a.mask = mask;
  a.order = order;
  a.tpi = tpi;
  a.per_frame = num_special + (a.cell ? (int64_t)a.hsy * a.wsx : 0);
  a.num_dst = tpi + (frames - 1) * a.per_frame;
  a.frames = (int)frames;
  a.ns = (int)num_special;
  a.sx = (int)sx;
  a.sy = (int)sy;
  hipLaunchKernelGGL(merge_order_kernel, dim3((unsigned)frames), dim3(kOrderThreads), 0,
                     (hipStream_t)stream, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    gpa_set_error("gpa_merge_order: launch failed: %s", hipGetErrorString(e));
    return GPA_E_LAUNCH;
  }
  return GPA_OK;
}

extern "C" size_t gpa_merge_plan_workspace_bytes(int64_t B, int64_t num_src) {
  if (B <= 0 || num_src <= 0) return 0;
  return radix_ws_bytes(B, num_src);     // either way's: the line depends on num_dst too
}

extern "C" int gpa_merge_plan(const void* node_max, int max_dtype, const int64_t* node_idx,
                              const int64_t* order, int64_t B, int64_t N, int64_t num_dst, int64_t r,
                              int64_t* edge, int64_t* dst_slot, int64_t* unm_abs, int64_t* src_abs,
                              float* size, int64_t* offsets, int64_t* tokens, void* workspace,
                              size_t workspace_bytes, void* stream) {
  static const char* fn = "gpa_merge_plan";
  gpa_clear_error();
  const int64_t ns = N - num_dst;
  if (B < 0 || N < 0 || num_dst < 0 || ns < 0 || r < 0 || r > ns) {
    gpa_set_error("%s: negative size, or more merged rows than sources", fn);
    return GPA_E_INVALID;
  }
  if (B == 0) return GPA_OK;
  if (num_dst == 0 && r > 0) {
    gpa_set_error("%s: %lld rows to merge and no destination", fn, (long long)r);
    return GPA_E_INVALID;
  }
  if (!offsets || (N > 0 && (!order || !size || !tokens)) ||
      (ns > 0 && (!node_max || !node_idx || !edge)) || (r > 0 && (!dst_slot || !src_abs)) ||
      (ns > r && !unm_abs)) {
    gpa_set_error("%s: null pointer", fn);
    return GPA_E_INVALID;
  }
  if (max_dtype != GPA_DTYPE_F32 && max_dtype != GPA_DTYPE_BF16 && max_dtype != GPA_DTYPE_F16) {
    gpa_set_error("%s: unknown dtype %d", fn, max_dtype);
    return GPA_E_INVALID;
  }
  if (N > 0x7ffff000LL || B > 65535) {
    gpa_set_error("%s: %lld x %lld tokens exceed the grid limit", fn, (long long)B, (long long)N);
    return GPA_E_UNSUPPORTED;
  }
  const bool rank = by_rank(B, ns, num_dst);
  const size_t need = rank ? rank_ws_bytes(B, ns) : radix_ws_bytes(B, ns);
  if (need && (!workspace || workspace_bytes < need || (uintptr_t)workspace % 16)) {
    gpa_set_error("%s: 16-byte aligned workspace of %zu bytes required, %zu given", fn, need,
                  workspace ? workspace_bytes : (size_t)0);
    return GPA_E_WORKSPACE;
  }
  PlanArgs a{};
  a.node_max = node_max;
  a.node_idx = node_idx;
  a.order = order;
  a.edge = edge;
  a.dst_slot = dst_slot;
  a.unm_abs = unm_abs;
  a.src_abs = src_abs;
  a.size = size;
  a.offsets = offsets;
  a.tokens = tokens;
  a.B = B;
  a.N = N;
  a.ns = (int)ns;
  a.num_dst = (int)num_dst;
  a.r = (int)r;
  // Kept rows carry the key num_dst and sort behind every destination; if
  // none is kept, the largest key is num_dst - 1.
  const uint64_t top = (uint64_t)(r < ns ? num_dst : num_dst > 0 ? num_dst - 1 : 0);
  a.passes = 1;
  while (a.passes < 4 && (top >> (8 * a.passes)) != 0) ++a.passes;
  a.blocks = (int)((ns + kTile - 1) / kTile);
  a.keys0 = (uint32_t*)workspace;
  if (!rank) {
    a.keys1 = a.keys0 + B * ns;
    a.vals0 = a.keys1 + B * ns;
    a.vals1 = a.vals0 + B * ns;
    a.counts = a.vals1 + B * ns;
  }
  hipStream_t s = (hipStream_t)stream;
  if (max_dtype == GPA_DTYPE_F32)
    plan_launch<float>(a, rank, s);
  else if (max_dtype == GPA_DTYPE_BF16)
    plan_launch<__bf16>(a, rank, s);
  else
    plan_launch<_Float16>(a, rank, s);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    gpa_set_error("%s: launch failed: %s", fn, hipGetErrorString(e));
    return GPA_E_LAUNCH;
  }
  return GPA_OK;
}
