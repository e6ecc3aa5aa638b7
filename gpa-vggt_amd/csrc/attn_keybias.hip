// Flash attention with a per-key additive bias for gfx950 (CDNA4), head_dim 64.
//
//   o[m,:]  = sum_n softmax_n(q_m.k_n * sm_scale + bias_n) v_n
//   lse[m]  = log2 sum_n 2^((q_m.k_n * sm_scale + bias_n) * log2 e)
//
// Semantics follow merging/fused_attention.py:70-127: scores in the exp2
// domain, fp32 online softmax, P rounded to the operand format for the P.V
// product, fp32 accumulation, log2 log-sum-exp output.  Every kernel is
// instantiated for bf16 and for fp16 operands (F16); only the MFMA opcode,
// the conversions and the offset constants differ.  Like the reference wrapper
// (fused_attention.py:159-160), a small pre-pass first writes the bias to a
// padded per-key buffer; here each 32-key tile gets a 144-byte record: the
// 32 values bias/sm_scale (-inf past N) and the tile's score bound below.
//
// Mapping onto CDNA4
//   * A workgroup owns 256 queries of one (batch, head): 4 waves of two
//     32-query blocks, <= 256 VGPRs each, so two workgroups share a CU (two
//     waves per SIMD).  Each K or V fragment read from LDS serves both of a
//     wave's blocks.
//   * One pass (attn_main_kernel), software-pipelined by one tile.  Every
//     wave runs with a fixed softmax offset certified on tile 0, or taken
//     from tile 0 and verified after the loop; a wave that can do neither
//     runs with a lazily moved offset (see there).
//   * K, V and the tile records stream through an LDS ring of 32-key tiles
//     filled by buffer_load ... lds (DMA into LDS, no staging registers)
//     several tiles ahead of the one being computed; keeping three tiles in
//     flight per workgroup is what hides the L2/HBM latency.
//   * Scores are computed transposed, S^T = K . Q^T, on
//     v_mfma_f32_32x32x16_bf16: a lane owns one query and 16 of the tile's
//     32 keys (the other 16 sit in lane^32), so the running max, the sum and
//     the rescale factor are per-lane scalars; the two halves meet through
//     v_permlane32_swap.  The accumulator starts from the tile's fp32
//     bias/sm_scale values (four broadcast LDS reads), so the MFMA chain
//     yields s = q.k + bias/sm_scale and x = s * (sm_scale*log2 e) - m is
//     one FMA.  Q stays unscaled: rounding q*sm_scale*log2(e) to bf16 would
//     perturb sharp logits by ~2^-9 of their size.
//   * P^T leaves the score MFMA already in the B-operand register layout of
//     the next MFMA, O^T = V^T . P^T, when the V^T A-operand enumerates keys
//     in the same order.  V stays row-major in LDS and the V^T operand is
//     read with ds_read_b64_tr_b16: within each 16-lane group, source lane
//     4v+a loads four features of key base+v and lane i receives feature
//     c0+i of keys base..base+3.  O^T keeps one query per lane, so a
//     rescale is a per-lane multiply.
//   * The softmax offset m only has to keep 2^(x-m) in range, since P is
//     stored in bf16, which has fp32's exponent range (fp16 P stops at 65504,
//     hence P <= 2^15 there): either a fixed offset derived from a
//     Cauchy-Schwarz bound on the scores, x <= c*(|q| max|k| + max
//     bias/sm_scale) (the tile records carry both maxima), or, where that
//     bound is too loose for the row, an offset that moves only when a tile's
//     exact max rises above m + kUp.  The result is the same softmax; only the
//     (arbitrary) offset differs from the reference's running max.
//   * Row sums add up the bf16 P the P.V product uses, on the matrix pipe:
//     v_mfma_f32_4x4x4_16b_bf16 with an all-ones A operand adds each lane's
//     four B values into its fp32 accumulator (four per block and tile).
//     The VALU is the busier unit of this kernel, and v_dot2_f32_bf16, the
//     other way to sum bf16 pairs, does not overlap an in-flight MFMA on
//     gfx950 (measured: 32 dot2 beside 16 MFMAs of 32x32x16 cost more than
//     running the two one after the other; fp32 adds, FMAs and the bf16
//     packing overlap it at ~95-98 %).  O is normalised by exactly the
//     weights it was built from, so two calls over a key partition combined
//     by their LSE give exactly the normalisation of one call over all keys.
//     The log-sum-exp is log2 of the sum of the bf16-rounded probabilities;
//     against the fp32 sum of the reference kernel (fused_attention.py:113)
//     every term differs by at most 2^-8 relative, so the LSE differs by at
//     most 2^-8 / ln 2 < 5.7e-3.
//   * LDS layouts are XOR-swizzled in 16-byte chunks so that the fragment
//     reads are free of bank conflicts under both 32- and 64-bank models;
//     the DMA lanes pick their global chunk so the swizzle costs nothing.
#include "gpa_common.h"

#include <math.h>

#include <mutex>

#include "attn_any_dim.h"
#include <type_traits>

namespace gpa {
namespace {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kBlk = 2;                       // 32-query blocks per wave
constexpr int kQPerWave = 32 * kBlk;
constexpr int kQPerWG = kWaves * kQPerWave;   // 256 queries per workgroup
constexpr int kKT = 32;                       // keys per tile
constexpr int kHD = 64;                       // head dim
constexpr float kMInit = -1.0e30f;            // finite initial offset (all -inf rows give 0)
// Offset window (log2 units).  Every P stays <= 2^kUp: for bf16 P (fp32's
// exponent range) 2^64 leaves row sums and O far below fp32's 2^128 for any
// key count and value size; fp16 P must stay below 65504.  A fixed offset is
// certified when each row's largest P is >= 2^-kDown: for bf16 2^-96 keeps
// every term that matters to 24 bits above fp32's normal range; for fp16 the
// largest P stays >= 2^-1, far from fp16's subnormals.  The lazily moved
// offset keeps the largest P in [1, 2^kUp].
template <bool F16> constexpr float kUp = F16 ? 15.0f : 64.0f;
template <bool F16> constexpr float kDown = F16 ? 1.0f : 96.0f;
// A wave whose rows the bound cannot certify may instead take the fixed
// offset m = x0 + kDown from tile 0 alone (its largest P is then >= 2^-kDown
// whatever the later tiles hold) and have it verified after the loop: only
// an overflow can go wrong, i.e. a later score more than kDown + ~100 (bf16;
// P is finite below 2^128 and sums of up to 2^24 keys stay finite) or
// kDown + 15.99 (fp16, P below 65504) log2 units above x0.  It does so when
// every row's tile-0 scores span at most kOptRange log2 units (for Gaussian
// scores the max over ~2^16 keys then sits about 0.55 times the largest
// span of the wave's rows above x0: ~143 against the ~192 bf16 allows, ~11
// against fp16's 16.99) and no key stands out: |q| (max_t c|k|_t -
// mean_t c|k|_t) + (max_t c b_t - mean_t c b_t) <= kOptOutlier over the
// per-tile maxima.  Other waves run the lazily moved offset from the start.
template <bool F16> constexpr float kOptRange = F16 ? 20.0f : 260.0f;
template <bool F16> constexpr float kOptOutlier = F16 ? 8.0f : 96.0f;
// A wave that fails that test on tile 0 looks at the first kMainAhead tiles
// (128 keys) instead and takes their max as x0 when their scores span at most
// kOptRange4 and the outlier term stays within kOptOutlier4.  Calibrated on
// N(0,1) q/k scaled up (68,700 keys, bias log counts): for fp16 the true max
// then sits at most ~15.6 log2 units above the 128-key max at x12 (0 of 2,048
// waves would overflow; all admitted), x14 admits 80 % of the waves of which
// 0.9 % overflow and are recomputed, x16 admits none.
template <bool F16> constexpr float kOptRange4 = F16 ? 34.0f : 320.0f;
template <bool F16> constexpr float kOptOutlier4 = F16 ? 12.0f : 96.0f;
constexpr int kRec = 36;                      // words per tile record
constexpr float kLog2e = 1.4426950408889634f;

struct AttnArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const float* recs;      // [B*H][ntiles][kRec] tile records
  const float* bounds;    // [B*H][kBoundWords] row bounds (row_bounds_kernel)
  uint8_t* flags;         // [B*H][gx][kWaves] per wave: 1 = the lazily moved offset ran
  uint16_t* o;
  float* lse;
  int H;
  int64_t M, N;
  int64_t q_sb, q_sh, q_sm, k_sb, k_sh, k_sn, v_sb, v_sh, v_sn, o_sb, o_sh, o_sm;
  int64_t lse_sb, lse_sh;
  uint32_t k_bytes, v_bytes, rec_bytes;  // extent of one (batch, head) slice
  float c;                                // sm_scale * log2(e)
  int o16;                                // O rows 16-byte aligned (16-byte stores)
  int no_bound;                           // records without key maxima: no score bound
  int fold;                               // form the row bounds here (at most kFoldTiles tiles)
};

// Another attention of the same queries over further keys, joined by LSE,
// contiguous and frame-major: o [B * M / P, H, P, 64], lse [B * M / P, H, P].
struct JoinArgs {
  const uint16_t* o;
  const float* lse;
  int P;
};

struct AttnJoinArgs {
  AttnArgs a;
  JoinArgs join;
};

struct RecArgs {
  const uint16_t* k;
  const void* bias;
  float* recs;
  int H;
  int64_t k_sb, k_sh, k_sn;
  int64_t sb, sh, sn;  // bias strides (0 = broadcast)
  int64_t N, ntiles;
  int64_t total;  // B * H * ntiles
  float mul;  // 1 / sm_scale
  float c;    // sm_scale * log2(e)
};

// K chunk swizzle: 16 consecutive keys reading one logical chunk hit 16
// distinct 16-byte bank groups (64 banks); any 8 consecutive keys hit 8
// (32 banks).
__device__ __forceinline__ int k_chunk(int key, int ch) {
  return ch ^ (key & 7) ^ ((key >> 3) & 1);
}

// V chunk swizzle for the transpose reads: the four keys of a 16-lane group
// and the two 8-byte halves of its chunks land in distinct banks.
__device__ __forceinline__ int v_chunk(int key, int ch) { return ch ^ ((key & 3) << 1); }

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t bits) {
  return __uint_as_float(bits << 16);
}

// DMA of 4 bytes per lane into LDS at lds + 4*lane.
__device__ __forceinline__ void dma4(__amdgpu_buffer_rsrc_t r, void* lds, uint32_t voff,
                                     uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      r, (__attribute__((address_space(3))) void*)lds, 4, voff, soff, 0, 0);
}

// DMA of 16 bytes per lane into LDS at lds + 16*lane.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, void* lds, uint32_t voff,
                                      uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      r, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, 0, 0);
}

// Wait until at most N vector-memory instructions of this wave are in flight
// (lgkm and export counters untouched).
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Tile records: one workgroup per kRecTiles consecutive 32-key tiles, eight
// lanes per key row (one 16-byte chunk each), so a wave's loads cover eight
// whole 128-byte rows.  Every lane issues its kRecTiles row loads (and bias
// loads) before it reduces any of them, which keeps 16 KB in flight per
// workgroup: with one tile per workgroup the kernel waited out one memory
// round trip per 4 KB.  The lanes of a key reduce its |k|^2; a tile's two
// maxima meet across the wave (xor 8, 16, 32) and then across the four
// waves in LDS.  Keys past N get bias -inf and |k| = 0; tiles past the last
// (batch, head) row are skipped.
constexpr int kRecTiles = 4;

// Bias bits of one key (uniform kind; no bias reads as 0).
template <int KIND>
__device__ __forceinline__ uint32_t bias_bits(const void* bias, int64_t off) {
  if constexpr (KIND == GPA_BIAS_F32) return static_cast<const uint32_t*>(bias)[off];
  else if constexpr (KIND == GPA_BIAS_NONE) return 0u;
  else return static_cast<const uint16_t*>(bias)[off];
}
template <int KIND>
__device__ __forceinline__ float bias_value(uint32_t bits) {
  if constexpr (KIND == GPA_BIAS_F32) return __uint_as_float(bits);
  else if constexpr (KIND == GPA_BIAS_BF16) return bf16_bits_to_f32((uint16_t)bits);
  else if constexpr (KIND == GPA_BIAS_F16) return (float)__builtin_bit_cast(_Float16, (uint16_t)bits);
  else return 0.f;
}

template <bool F16, int KIND>
__global__ __launch_bounds__(256) void tile_records_kernel(RecArgs a) {
  __shared__ float part[kRecTiles][2][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int j = tid >> 3, ch = tid & 7;                // key of the tile, 16-byte chunk
  const int64_t tile0 = (int64_t)blockIdx.x * kRecTiles;
  const int64_t row0 = tile0 / a.ntiles;
  int64_t t = tile0 - row0 * a.ntiles, hb = row0 % a.H, bb = row0 / a.H;
  // All loads first, without branches: a key that does not exist (past N,
  // or in a tile past the last row) reads element 0 of K and of the bias
  // instead and is masked afterwards.
  bf16x8 kv[kRecTiles];
  uint32_t xb[kRecTiles];
  bool live[kRecTiles];
#pragma unroll
  for (int u = 0; u < kRecTiles; ++u) {
    const int64_t n = t * kKT + j;
    live[u] = tile0 + u < a.total && n < a.N;
    const int64_t koff = live[u] ? bb * a.k_sb + hb * a.k_sh + n * a.k_sn : 0;
    const int64_t boff = live[u] ? bb * a.sb + hb * a.sh + n * a.sn : 0;
    kv[u] = *reinterpret_cast<const bf16x8*>(a.k + koff + ch * 8);
    xb[u] = bias_bits<KIND>(a.bias, boff);
    if (++t == a.ntiles) {
      t = 0;
      if (++hb == a.H) {
        hb = 0;
        ++bb;
      }
    }
  }
#pragma unroll
  for (int u = 0; u < kRecTiles; ++u) {
    const float x = live[u] ? bias_value<KIND>(xb[u]) * a.mul : -INFINITY;
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = half_to_f32<F16>(kv[u][e]);
      ss = __builtin_fmaf(f, f, ss);
    }
#pragma unroll
    for (int w = 1; w < 8; w <<= 1) ss += __shfl_xor(ss, w);
    float kmax = live[u] ? __builtin_sqrtf(ss) : 0.f, xmax = x;
#pragma unroll
    for (int w = 8; w < 64; w <<= 1) {
      kmax = fmaxf(kmax, __shfl_xor(kmax, w));
      xmax = fmaxf(xmax, __shfl_xor(xmax, w));
    }
    if (lane == 0) {
      part[u][0][wave] = kmax;
      part[u][1][wave] = xmax;
    }
    if (ch == 0 && tile0 + u < a.total) a.recs[(tile0 + u) * kRec + j] = x;
  }
  __syncthreads();
  constexpr int kTail = kRec - kKT;                    // words after the 32 biases
  if (tid < kRecTiles * kTail) {
    const int u = tid / kTail, r = tid % kTail;
    if (tile0 + u < a.total) {
      const float km = fmaxf(fmaxf(part[u][0][0], part[u][0][1]), fmaxf(part[u][0][2], part[u][0][3]));
      const float xm = fmaxf(fmaxf(part[u][1][0], part[u][1][1]), fmaxf(part[u][1][2], part[u][1][3]));
      a.recs[(tile0 + u) * kRec + kKT + r] = r == 0 ? a.c * km : r == 1 ? a.c * xm : 0.f;
    }
  }
}

// Per (batch, head): the maxima over its tiles of c*max|k| and
// c*max bias/sm_scale, so c*(|q| K + B) bounds every score of a query, and
// the means over its tiles of the same two words (how far the largest key
// norm and the largest bias stand out from the rest of the keys).
// kBoundWords floats per (batch, head).
constexpr int kBoundWords = 4;
// Up to this many tiles (8,192 keys) every wave of the attention forms them
// from the records itself, which saves the launch: 16 heads, 2,748 queries and
// 1,703 keys 38.4 -> 36.7 us, 5,496 x 2,361 76.6 -> 75.4 us, 21,984 x 7,721
// within 0.1 %.  It delays every workgroup a little, though, so the line lies
// at two rounds of the chip's 512 places: 40 fp16 frames (3,840 workgroups of
// 43 tiles) took 352 us so and take 348 us with the launch.  (The records and
// the bounds by one workgroup per head in one launch took 6 us more than the
// two launches.)
constexpr int kFoldLoads = 4, kFoldTiles = 64 * kFoldLoads;
constexpr int64_t kFoldGrid = 1024;
__global__ __launch_bounds__(256) void row_bounds_kernel(const float* recs, float* bounds,
                                                         int64_t ntiles) {
  __shared__ float part[4][4];
  const float* r = recs + (int64_t)blockIdx.x * ntiles * kRec;
  float kb = 0.f, bb = -INFINITY, ks = 0.f, bs = 0.f;
  for (int64_t t = threadIdx.x; t < ntiles; t += 256) {
    const float kt = r[t * kRec + kKT], bt = r[t * kRec + kKT + 1];
    kb = fmaxf(kb, kt);
    bb = fmaxf(bb, bt);
    ks += kt;
    bs += bt;
  }
#pragma unroll
  for (int w = 1; w < 64; w <<= 1) {
    kb = fmaxf(kb, __shfl_xor(kb, w));
    bb = fmaxf(bb, __shfl_xor(bb, w));
    ks += __shfl_xor(ks, w);
    bs += __shfl_xor(bs, w);
  }
  if ((threadIdx.x & 63) == 0) {
    part[0][threadIdx.x >> 6] = kb;
    part[1][threadIdx.x >> 6] = bb;
    part[2][threadIdx.x >> 6] = ks;
    part[3][threadIdx.x >> 6] = bs;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float* out = bounds + (int64_t)kBoundWords * blockIdx.x;
    out[0] = fmaxf(fmaxf(part[0][0], part[0][1]), fmaxf(part[0][2], part[0][3]));
    out[1] = fmaxf(fmaxf(part[1][0], part[1][1]), fmaxf(part[1][2], part[1][3]));
    out[2] = ((part[2][0] + part[2][1]) + (part[2][2] + part[2][3])) / (float)ntiles;
    out[3] = ((part[3][0] + part[3][1]) + (part[3][2] + part[3][3])) / (float)ntiles;
  }
}

// Workgroup barrier that does not drain the vector-memory counter: the
// in-flight DMAs of later tiles must stay in flight across it (the explicit
// wait_vm before it covers the tile that has to be complete).  The memory
// clobber keeps the compiler from moving LDS accesses across it, and
// lgkmcnt(0) retires this wave's LDS reads before any slot is refilled.
__device__ __forceinline__ void tile_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Tile records of a joined call without bias, bf16 (unjoined ones need none:
// attn_plain_kernel): bias/sm_scale = 0 for the keys, -inf past N, and no key
// maxima, so the kernel has no score bound and every wave takes the tile-0
// offset or the lazily moved one.  Writing these costs nothing like reading
// every key.  Also zeroes the row-bound words the kernel reads.
__global__ __launch_bounds__(256) void fill_records_kernel(float* recs, float* bounds,
                                                           int64_t ntiles, int64_t N,
                                                           int64_t total, int64_t rows) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < total * kRec) {
    const int64_t t = i / kRec, w = i - t * kRec;
    const int64_t n = (t % ntiles) * kKT + w;
    recs[i] = (w < kKT && n >= N) ? -INFINITY : 0.f;
  }
  if (i < rows * kBoundWords) bounds[i] = 0.f;
}

// The attention kernel: software-pipelined by one tile.
//
// On gfx950 a wave's MFMAs overlap its own VALU work well (measured: 16
// MFMAs of 32x32x16 interleaved with a tile's softmax in one wave run at
// ~78 % of the MFMA rate) but another wave's only weakly (~40 % when one
// wave on a SIMD issues the MFMAs and another the VALU work).  So each
// iteration t gives the wave independent work for both units:
//   MFMA  S(t+1) = K(t+1).Q^T + bias(t+1) for both query blocks (8), then
//         O += V(t)^T . P(t) per block as its P is ready (8), and the row
//         sums of P(t) (8 small 4x4x4 MFMAs)
//   VALU  P(t) = 2^(S(t) c - m) in bf16 (32 FMA + 32 exp + 16 packs)
// and sched_group_barrier interleaves them, one MFMA to three VALU
// instructions, after the iteration's LDS reads.  Only the last block's
// P.V product has no VALU work beside it.
//
// The softmax offset.  B = c*(|q| max|k| + max bias/sm_scale) over all keys
// bounds every score of a row (Cauchy-Schwarz).  From tile 0's exact row
// max x0 the wave takes the fixed offset m = max(B - kUp, x0): no score can
// then produce P above 2^kUp, and the wave is certified when every row has
// x0 >= m - kDown, i.e. the row's largest P is at least 2^-kDown.  A
// certified wave runs the loop with no max, rescale or branch at all.  A wave
// that cannot certify (B far above the row's real scores: sharp logits, or
// fp16's narrow window, which LayerNorm-scaled q and k already exceed) runs
// the same loop with the tile-0 offset m = x0 + kDown when its tile-0 scores
// are narrow and no key stands out (kOptRange, kOptOutlier): its largest P
// is then >= 2^-kDown, and after the loop the row sums and O are checked for
// an overflow (a later score more than ~192 / 17 log2 units above x0).  If a
// wave of the workgroup overflowed, the workgroup streams the keys again and
// every live wave recomputes its rows with the lazily moved offset.  Waves
// outside both cases run that lazy loop from the start: m starts at x0 and,
// per tile, S(t), its exact row max, a wave-uniform branch that rescales O
// and the row sums only where that max exceeds m + kUp, then P(t) and its
// P.V product.  That loop is not pipelined (S(t) and P(t) in the same
// iteration), so it holds fewer live registers than the certified loop and
// leaves its register allocation and schedule as they are (compared opcode
// by opcode).  All loops issue the same DMAs, waits and barriers.  The
// per-wave flag records what ran: bit 0 the output came from the lazy loop,
// bit 1 the wave took the tile-0 offset, bit 2 the workgroup streamed twice.
//
// Five ring slots keep tile t (V), tile t+1 (K, bias) and the three tiles
// in flight; the DMA of tile t+4 refills the slot of tile t-1.  Every wave
// issues the record DMA (64 lanes x 4 bytes, so a slot's record area is
// 256 bytes, of which the first 144 are the record): wave 0 into the slot,
// the others into a scratch area nobody reads, so no wave-dependent branch
// splits an iteration; lanes outside the record read zeros by range.  The
// unrolled iterations then form one basic block, in which the pure
// arithmetic of an iteration could float down to its consumers in the next
// one; an empty asm that takes the iteration's results as operands keeps it
// inside.  At most 256 VGPRs, two waves per SIMD.
constexpr int kMainSlots = 5;
constexpr int kMainAhead = kMainSlots - 1;  // tiles issued ahead of the one being softmaxed

struct alignas(16) MainTile {
  uint16_t k[kKT * kHD];
  uint16_t v[kKT * kHD];
  float rec[64];
};

// Records of a call without bias are zeros, but for the keys past N of the last
// tile: row N % 32 of this table, -inf from there on (row 0: a whole tile).
struct TailRecords {
  float w[kKT][kRec];
};
constexpr TailRecords tail_records() {
  TailRecords t{};
  for (int r = 1; r < kKT; ++r)
    for (int k = r; k < kKT; ++k) t.w[r][k] = -__builtin_inff();
  return t;
}
__device__ const TailRecords kTail = tail_records();

// PLAIN: no bias and no score bound (bf16), so no records in memory.
template <bool F16, bool JOIN, bool PLAIN>
__device__ __forceinline__ void attn_main_body(const AttnArgs& p) {
  __shared__ MainTile ring0, ring1, ring2, ring3, ring4;
  __shared__ float rec_sink[64];
  __shared__ uint32_t wg_fail[kWaves];   // per wave: its tile-0 offset overflowed
  MainTile* const ring[kMainSlots] = {&ring0, &ring1, &ring2, &ring3, &ring4};

  const int tid = threadIdx.x;
  const int lane = tid & 63, hi = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // XCD-aware order: the hardware deals consecutive workgroups round-robin
  // to the 8 XCDs, so each XCD is given a contiguous range of (batch-head,
  // query block) items instead, and the query blocks of one batch-head share
  // that XCD's L2 for their K and V (own-frame attention: 6 %).
  int qb, bh;
  {
    const uint32_t T = gridDim.x * gridDim.y, L = blockIdx.y * gridDim.x + blockIdx.x;
    const uint32_t q8 = T / 8, r8 = T % 8, x = L % 8;
    const uint32_t item = x * q8 + (x < r8 ? x : r8) + L / 8;
    qb = (int)(item % gridDim.x);
    bh = (int)(item / gridDim.x);
  }
  const int64_t b = bh / p.H, h = bh % p.H;
  uint8_t* const flag_row = p.flags + ((int64_t)bh * gridDim.x + qb) * kWaves;
  const int64_t q_base = (int64_t)qb * kQPerWG + wave * kQPerWave + l32;
  const float c = p.c;
  const uint16_t* Q = p.q + b * p.q_sb + h * p.q_sh;
  const uint16_t* K = p.k + b * p.k_sb + h * p.k_sh;
  const uint16_t* V = p.v + b * p.v_sb + h * p.v_sh;
  const float* R = PLAIN ? kTail.w[(int)p.N & (kKT - 1)] : p.recs + (int64_t)bh * (p.rec_bytes / 4);
  // The output bases, formed here so that only two pointers (not five
  // 64-bit strides) stay live in SGPRs until the epilogue.
  uint16_t* O = p.o + b * p.o_sb + h * p.o_sh;
  float* LSE = !JOIN && p.lse ? p.lse + b * p.lse_sb + h * p.lse_sh : nullptr;
  const int o_sm = (int)p.o_sm;
  if constexpr (JOIN) asm volatile("" : "+s"(O));
  else asm volatile("" : "+s"(O), "+s"(LSE));

  const float* const rb = p.bounds + (int64_t)kBoundWords * bh;
  float row_k = 0.f, row_b = 0.f, row_kmean = 0.f, row_bmean = 0.f;
  if constexpr (PLAIN) {
  } else if (p.fold) {
    const int nt = (int)((p.N + kKT - 1) / kKT);
    float kb = 0.f, bb = -INFINITY, ks = 0.f, bs = 0.f;
    u32x2 w2[kFoldLoads];
#pragma unroll
    for (int i = 0; i < kFoldLoads; ++i)
      w2[i] = *reinterpret_cast<const u32x2*>(R + (lane + 64 * i < nt ? lane + 64 * i : 0) * kRec + kKT);
#pragma unroll
    for (int i = 0; i < kFoldLoads; ++i)
      if (lane + 64 * i < nt) {
        const float kt = __uint_as_float(w2[i][0]), bt = __uint_as_float(w2[i][1]);
        kb = fmaxf(kb, kt);
        bb = fmaxf(bb, bt);
        ks += kt;
        bs += bt;
      }
#pragma unroll
    for (int w = 1; w < 64; w <<= 1) {
      kb = fmaxf(kb, __shfl_xor(kb, w));
      bb = fmaxf(bb, __shfl_xor(bb, w));
      ks += __shfl_xor(ks, w);
      bs += __shfl_xor(bs, w);
    }
    auto uniform = [](float x) {                 // to SGPRs
      return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x)));
    };
    row_k = uniform(kb);
    row_b = uniform(bb);
    row_kmean = uniform(ks / (float)nt);
    row_bmean = uniform(bs / (float)nt);
  } else {
    row_k = rb[0];
    row_b = rb[1];
    row_kmean = rb[2];
    row_bmean = rb[3];
  }

  // Q^T as the B-operand of S^T = K . Q^T: in block j the lane supplies
  // query q_base + 32 j, features 16*ks + 8*hi .. +8.  Only the loads here:
  // |q| (for the bound) is formed after the prologue's tile DMAs are issued,
  // so that both blocks' Q loads and the first tiles are in flight together.
  // Formed right after each block's loads, it made the compiler wait for
  // them before issuing anything else: three memory round trips in a row
  // before the first tile (about 3 us of a 48 us own-frame workgroup).
  bf16x8 qf[kBlk][4];
  float q_norm[kBlk];
#pragma unroll
  for (int j = 0; j < kBlk; ++j) {
    const int64_t row = q_base + 32 * j;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      qf[j][ks] = row < p.M ? *reinterpret_cast<const bf16x8*>(Q + row * p.q_sm + ks * 16 + hi * 8)
                            : bf16x8{};
  }
  __builtin_amdgcn_sched_barrier(0);

  const __amdgpu_buffer_rsrc_t krs = make_rsrc(K, p.k_bytes);
  const __amdgpu_buffer_rsrc_t vrs = make_rsrc(V, p.v_bytes);
  const __amdgpu_buffer_rsrc_t rrs = make_rsrc(R, PLAIN ? kRec * 4u : p.rec_bytes);
  const uint32_t k_row = (uint32_t)p.k_sn * 2u, v_row = (uint32_t)p.v_sn * 2u;
  const int slot = wave * 64 + lane;
  const int s_key = slot >> 3, s_pc = slot & 7;
  const uint32_t k_voff = s_key * k_row + k_chunk(s_key, s_pc) * 16;
  const uint32_t v_voff = s_key * v_row + v_chunk(s_key, s_pc) * 16;
  // The record DMA moves 4 bytes per lane: wave 0's first 36 lanes fetch the
  // 144-byte record; every other lane points past the descriptor's range
  // (2^30 > any record row), so it lands zeros without touching memory.
  const uint32_t rec_voff = (wave == 0 && lane < kRec) ? (uint32_t)lane * 4u : 0x40000000u;
  const int ntiles = (int)((p.N + kKT - 1) / kKT);
  auto issue = [&](int t, MainTile& T) {
    const uint32_t n0 = (uint32_t)t * kKT;
    dma16(krs, &T.k[wave * 512], k_voff, n0 * k_row);
    dma16(vrs, &T.v[wave * 512], v_voff, n0 * v_row);
    float* dst = wave == 0 ? &T.rec[0] : &rec_sink[0];   // wave-uniform M0, no branch
    if constexpr (PLAIN)       // every tile but the last lands zeros: an empty range
      dma4(make_rsrc(R, t == ntiles - 1 ? kRec * 4u : 0u), dst, rec_voff, 0);
    else
      dma4(rrs, dst, rec_voff, (uint32_t)t * (kRec * 4));
  };
  // A tile has landed once at most the DMAs of the NT tiles issued after it
  // (three instructions per tile) are outstanding.
  auto wait_tiles = [&](auto nt) {
    constexpr int NT = decltype(nt)::value;
    wait_vm<3 * NT>();
  };

  int k_off[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) k_off[ks] = l32 * kHD + (k_chunk(l32, 2 * ks + hi) << 3);
  int v_base[2];
#pragma unroll
  for (int db = 0; db < 2; ++db) {
    const int key = 4 * hi + ((lane & 15) >> 2);
    const int a = lane & 3;
    const int ch = db * 4 + ((lane >> 4) & 1) * 2 + (a >> 1);
    v_base[db] = key * kHD + (v_chunk(key, ch) << 3) + (a & 1) * 4;
  }

  float m_off[kBlk];
  f32x4 l_acc[kBlk];
  f32x16 o_acc[kBlk][2];
#pragma unroll
  for (int j = 0; j < kBlk; ++j) {
    l_acc[j] = f32x4{};
    o_acc[j][0] = f32x16{};
    o_acc[j][1] = f32x16{};
  }

  // S(T) for both blocks; the accumulators start from the keys' bias values.
  auto scores = [&](const MainTile& T, f32x16 (&sv)[kBlk]) {
    f32x16 bias16;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 bv = *reinterpret_cast<const f32x4*>(&T.rec[8 * g + 4 * hi]);
      bias16[4 * g + 0] = bv[0];
      bias16[4 * g + 1] = bv[1];
      bias16[4 * g + 2] = bv[2];
      bias16[4 * g + 3] = bv[3];
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const bf16x8 kf = *reinterpret_cast<const bf16x8*>(&T.k[k_off[ks]]);
#pragma unroll
      for (int j = 0; j < kBlk; ++j)
        sv[j] = mfma32x32x16_t<F16>(kf, qf[j][ks], ks == 0 ? bias16 : sv[j]);
    }
  };
  // V^T fragments of a tile (shared by both blocks).
  auto read_v = [&](const MainTile& T, bf16x8 (&vf)[2][2]) {
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        typedef short i16x4 __attribute__((ext_vector_type(4)));
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) i16x4*)&T.v[v_base[db] + 1024 * s]);
        const i16x4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) i16x4*)&T.v[v_base[db] + 1024 * s + 512]);
        const bf16x4 l4 = __builtin_bit_cast(bf16x4, lo), u4 = __builtin_bit_cast(bf16x4, up);
        vf[db][s] = bf16x8{l4[0], l4[1], l4[2], l4[3], u4[0], u4[1], u4[2], u4[3]};
      }
  };
  // Exact row max of a block's scores, in log2 units: the row's 16 keys in
  // this lane and 16 in lane^32.
  auto row_max = [&](const f32x16& x) {
    float mx = fmaxf(fmaxf(x[0], x[1]), x[2]);
#pragma unroll
    for (int r = 3; r < 15; r += 2) mx = fmaxf(fmaxf(mx, x[r]), x[r + 1]);
    mx = fmaxf(mx, x[15]);
    return max_halves(mx) * c;
  };
  // Min over the row's live scores (keys past N score -inf), in log2 units.
  auto row_min = [&](const f32x16& x) {
    float mn = INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mn = x[r] > -INFINITY ? fminf(mn, x[r]) : mn;
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mn), __float_as_uint(mn),
                                                     false, false);
    return fminf(__uint_as_float(sw[0]), __uint_as_float(sw[1])) * c;
  };
  // P = 2^(S c - m) of one block in bf16, its row sums, then O += V^T . P.
  const __bf16 one = f32_to_half<F16>(1.0f);
  const bf16x4 ones4 = {one, one, one, one};
  auto softmax_pv = [&](const f32x16& sv, int j, const bf16x8 (&vf)[2][2]) {
    const float neg_m = -m_off[j];
    bf16x8 pb[2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      // Source order steers the compiler here.  fp16: the eight exp2 first,
      // then the packs, or most packs sit right after their exp2 and take a
      // wait state each (90 s_nop per five iterations against 23).  bf16:
      // pairwise, or the packs get split into single conversions and perms.
      if constexpr (F16) {
        float pe[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
          pe[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[8 * half + e], c, neg_m));
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const bf16x2 pv2 = pack2<F16>(pe[e], pe[e + 1]);
          pb[half][e] = pv2[0];
          pb[half][e + 1] = pv2[1];
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[8 * half + e], c, neg_m));
          const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[8 * half + e + 1], c, neg_m));
          const bf16x2 pv2 = pack2<F16>(p0, p1);
          pb[half][e] = pv2[0];
          pb[half][e + 1] = pv2[1];
        }
      }
      const bf16x4 lo = {pb[half][0], pb[half][1], pb[half][2], pb[half][3]};
      const bf16x4 up = {pb[half][4], pb[half][5], pb[half][6], pb[half][7]};
      l_acc[j] = mfma4x4x4_t<F16>(ones4, lo, l_acc[j]);
      l_acc[j] = mfma4x4x4_t<F16>(ones4, up, l_acc[j]);
    }
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int s = 0; s < 2; ++s) o_acc[j][db] = mfma32x32x16_t<F16>(vf[db][s], pb[s], o_acc[j][db]);
  };

  f32x16 s_cur[kBlk], s_nxt[kBlk];
  auto pin_iteration = [&]() {
#pragma unroll
    for (int j = 0; j < kBlk; ++j) {
      asm volatile("" : "+v"(s_nxt[j]), "+v"(l_acc[j]));
      asm volatile("" : "+v"(o_acc[j][0]), "+v"(o_acc[j][1]));
    }
  };

  // A wave whose 64 queries all lie past M (waves 2 and 3 of the last query
  // block of a batch-head when M mod 256 <= 128, e.g. 94 of 1,374) only
  // carries its share of every tile's DMA: the same DMAs, waits and barriers
  // as a live wave, no MFMA or softmax work, so the live wave sharing its
  // SIMD gets the matrix pipe to itself.  Wave-uniform branch, taken before
  // the live path starts.  Should the workgroup stream the keys a second
  // time (see the verification below), such a wave takes the live waves'
  // recompute path on its zero-filled queries, whose rows are never stored:
  // a second copy of the stream loop here costs the whole kernel SGPR and
  // VGPR spills.
  const bool dead = (int64_t)qb * kQPerWG + wave * kQPerWave >= p.M;
  bool fixed = false, opt = false;
  if (dead) {
#pragma unroll
    for (int i = 0; i < kMainAhead; ++i) issue(i, *ring[i]);
    wait_tiles(std::integral_constant<int, kMainAhead - 1>{});
    tile_barrier();
    wait_tiles(std::integral_constant<int, 0>{});
    tile_barrier();
    auto carry = [&](const int t, MainTile& Tissue) {
      issue(t + kMainAhead, Tissue);
      wait_tiles(std::integral_constant<int, kMainAhead - 2>{});
      tile_barrier();
    };
    int t = 0;
    for (; t + kMainSlots <= ntiles; t += kMainSlots) {
#pragma unroll
      for (int u = 0; u < kMainSlots; ++u) carry(t + u, *ring[(u + kMainAhead) % kMainSlots]);
    }
#pragma unroll
    for (int u = 0; u < kMainSlots - 1; ++u)
      if (t < ntiles) {
        carry(t, *ring[(u + kMainAhead) % kMainSlots]);
        ++t;
      }
  } else {
  // Prologue: tiles 0 .. kMainAhead-1 in flight behind the Q loads; |q|;
  // S(0) and the certification.
#pragma unroll
  for (int i = 0; i < kMainAhead; ++i) issue(i, *ring[i]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < kBlk; ++j) {
    float ss = 0.f;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float f = half_to_f32<F16>(qf[j][ks][e]);
        ss = __builtin_fmaf(f, f, ss);
      }
    q_norm[j] = __builtin_sqrtf(sum_halves(ss));
  }
  wait_tiles(std::integral_constant<int, kMainAhead - 1>{});
  tile_barrier();
  scores(*ring[0], s_cur);
  bool bad = false;
  float x0s[kBlk];
#pragma unroll
  for (int j = 0; j < kBlk; ++j) {
    x0s[j] = row_max(s_cur[j]);
    // (A value of its own in every kernel, not one end of an FMA with kDown in
    // the one that has no other use for it: the same offset, the same P.)
    asm volatile("" : "+v"(x0s[j]));
    m_off[j] = fmaxf(__builtin_fmaf(q_norm[j], row_k, row_b) - kUp<F16>, x0s[j]);
    bad = bad || !(x0s[j] >= m_off[j] - kDown<F16>);     // NaN scores fail too
  }
  // (Without the key maxima there is no bound to certify anything with.)
  fixed = !PLAIN && !p.no_bound && __builtin_amdgcn_ballot_w64(bad) == 0;
  float lo[kBlk], outl[kBlk];
  if (!fixed) {
    // The tile-0 offset, taken where tile 0's scores are narrow and no key
    // stands out (so that an overflow is unlikely); verified after the loop.
    bool wide = false;
#pragma unroll
    for (int j = 0; j < kBlk; ++j) {
      lo[j] = row_min(s_cur[j]);
      outl[j] = __builtin_fmaf(q_norm[j], row_k - row_kmean, row_b - row_bmean);
      wide = wide || !(x0s[j] > -INFINITY && x0s[j] < INFINITY) ||
             !(x0s[j] - lo[j] <= kOptRange<F16>) || !(outl[j] <= kOptOutlier<F16>);
    }
    opt = __builtin_amdgcn_ballot_w64(wide) == 0;
#pragma unroll
    for (int j = 0; j < kBlk; ++j)
      m_off[j] = opt ? x0s[j] + kDown<F16> : kMInit;      // lazy: the first tile moves it
  }
  // All kMainAhead tiles have landed past this barrier (every wave path waits
  // for all of them here), so a wave may read any of them.
  wait_tiles(std::integral_constant<int, 0>{});
  tile_barrier();
  if (!fixed && !opt) {
    // The tile-0 test failed: widen the sample to the first kMainAhead tiles
    // (already in LDS; s_nxt is free until the loop) and take their row max
    // as the offset if the scores seen so far are narrow enough (kOptRange4,
    // kOptOutlier4); still verified after the loop.
    float x4[kBlk];
#pragma unroll
    for (int j = 0; j < kBlk; ++j) x4[j] = x0s[j];
#pragma unroll
    for (int i = 1; i < kMainAhead; ++i)
      if (i < ntiles) {
        scores(*ring[i], s_nxt);
#pragma unroll
        for (int j = 0; j < kBlk; ++j) {
          x4[j] = fmaxf(x4[j], row_max(s_nxt[j]));
          lo[j] = fminf(lo[j], row_min(s_nxt[j]));
        }
      }
    bool wide = false;
#pragma unroll
    for (int j = 0; j < kBlk; ++j)
      wide = wide || !(x4[j] > -INFINITY && x4[j] < INFINITY) ||
             !(x4[j] - lo[j] <= kOptRange4<F16>) || !(outl[j] <= kOptOutlier4<F16>);
    opt = __builtin_amdgcn_ballot_w64(wide) == 0;
    if (opt) {
#pragma unroll
      for (int j = 0; j < kBlk; ++j) m_off[j] = x4[j] + kDown<F16>;
    }
  }
  }

  // Iteration t: refill the slot of tile t-1 with tile t+kMainAhead; S(t+1)
  // beside the softmax of S(t); P.V of tile t; tile t+2 lands by its end.
  // (For t = ntiles-1 the S of the tile past the end is computed from
  // zero-filled K and records and never used.)
  auto iter = [&](const int t, const MainTile& Tcur, const MainTile& Tnext, MainTile& Tissue) {
    __builtin_amdgcn_sched_barrier(0);
    issue(t + kMainAhead, Tissue);
    scores(Tnext, s_nxt);
    bf16x8 vf[2][2];
    read_v(Tcur, vf);
    softmax_pv(s_cur[0], 0, vf);
    softmax_pv(s_cur[1], 1, vf);
    __builtin_amdgcn_sched_group_barrier(0x100, 16, 0);   // the 16 LDS reads first
#pragma unroll
    for (int i = 0; i < 24; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
      __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);  // three VALU
    }
    pin_iteration();
    wait_tiles(std::integral_constant<int, kMainAhead - 2>{});
    tile_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < kBlk; ++j) s_cur[j] = s_nxt[j];
  };
  // The lazily moved offset: tile t whole (its K and V are both resident in
  // iteration t), with the same DMA, wait and barrier as `iter`.
  auto lazy_iter = [&](const int t, const MainTile& Tcur, MainTile& Tissue) {
    issue(t + kMainAhead, Tissue);
    f32x16 sv[kBlk];
    scores(Tcur, sv);
    bf16x8 vf[2][2];
    read_v(Tcur, vf);
    // (One branch level per block: nested ones make the register allocator
    // copy the O accumulators on every tile.)
#pragma unroll
    for (int j = 0; j < kBlk; ++j) {
      const float mx = row_max(sv[j]);
      if (__builtin_amdgcn_ballot_w64(mx > m_off[j] + kUp<F16>) != 0) {
        const float m_new = mx > m_off[j] + kUp<F16> ? mx : m_off[j];
        const float alpha = __builtin_amdgcn_exp2f(m_off[j] - m_new);
        m_off[j] = m_new;
        l_acc[j] *= alpha;
        o_acc[j][0] *= alpha;
        o_acc[j][1] *= alpha;
      }
    }
    softmax_pv(sv[0], 0, vf);
    softmax_pv(sv[1], 1, vf);
    wait_tiles(std::integral_constant<int, kMainAhead - 2>{});
    tile_barrier();
  };
  // Unrolled by the ring size, so every slot is a compile-time LDS object
  // (the waitcnt pass can then tell a slot being read from one being filled).
  auto run = [&](auto lazy) {
    constexpr bool LAZY = decltype(lazy)::value;
    auto step = [&](const int t, const int u) {
      if constexpr (LAZY)
        lazy_iter(t, *ring[u], *ring[(u + kMainAhead) % kMainSlots]);
      else
        iter(t, *ring[u], *ring[(u + 1) % kMainSlots], *ring[(u + kMainAhead) % kMainSlots]);
    };
    int t = 0;
    for (; t + kMainSlots <= ntiles; t += kMainSlots) {
#pragma unroll
      for (int u = 0; u < kMainSlots; ++u) step(t + u, u);
    }
#pragma unroll
    for (int u = 0; u < kMainSlots - 1; ++u)
      if (t < ntiles) {
        step(t, u);
        ++t;
      }
  };
  if (!dead) {
    if (fixed || opt)
      run(std::false_type{});
    else
      run(std::true_type{});
  }
  // Drain the DMAs still in flight (before the ring is reused or the
  // workgroup exits).
  wait_vm<0>();

  // Verification of the tile-0 offset: any P that overflowed made its row
  // sum infinite, a product that overflowed made O infinite (NaN counts as
  // a failure too).  If a wave failed, the whole workgroup streams the keys
  // again and every live wave recomputes its rows with the lazily moved
  // offset (the ring is shared, so the others carry their share of the
  // DMAs); the first results are discarded.
  bool fail = false;
  if (opt) {
#pragma unroll
    for (int j = 0; j < kBlk; ++j) {
      fail = fail || !(sum_halves(l_acc[j][0]) < INFINITY);
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) fail = fail || !(fabsf(o_acc[j][db][r]) < INFINITY);
    }
  }
  const bool fail_w = __builtin_amdgcn_ballot_w64(fail) != 0;   // every lane's verdict
  if (lane == 0) wg_fail[wave] = fail_w ? 1u : 0u;
  tile_barrier();
  const bool rerun = __builtin_amdgcn_readfirstlane(wg_fail[0] | wg_fail[1] | wg_fail[2] |
                                                    wg_fail[3]) != 0;
  if (rerun) {
#pragma unroll
    for (int j = 0; j < kBlk; ++j) {
      l_acc[j] = f32x4{};
      o_acc[j][0] = f32x16{};
      o_acc[j][1] = f32x16{};
      m_off[j] = kMInit;
    }
#pragma unroll
    for (int i = 0; i < kMainAhead; ++i) issue(i, *ring[i]);
    wait_tiles(std::integral_constant<int, kMainAhead - 1>{});
    tile_barrier();
    wait_tiles(std::integral_constant<int, 0>{});
    tile_barrier();
    run(std::true_type{});
    wait_vm<0>();
    tile_barrier();
  }
  // Flag bits: 1 = the output comes from the lazily moved offset, 2 = the
  // wave took the tile-0 offset, 4 = its workgroup streamed the keys twice
  // (a wave without queries: 0 or 4).
  if (dead) {
    if (lane == 0) flag_row[wave] = rerun ? 4 : 0;
    return;
  }
  if (lane == 0)
    flag_row[wave] = (uint8_t)((rerun || !(fixed || opt) ? 1 : 0) | (opt ? 2 : 0) | (rerun ? 4 : 0));

  // O goes through LDS so that every store writes whole 128-byte rows:
  // eight rows of 16 bytes per lane per instruction instead of 8 bytes in
  // each of 32 rows (the strided stores took ~2 us per workgroup to issue).
  // Wave w stages its 64 rows in ring slot w (8 KB of its 8.25 KB), free once
  // every wave has drained its DMAs (the barrier).  Row r of the wave (block
  // r / 32, query row r % 32) keeps its 16-byte chunk c at chunk c ^ (r & 7):
  // the writes of one instruction meet at most two to a bank, the row reads
  // not at all.  A wave's LDS operations run in order, so the reads need no
  // further barrier.  (The verdict barrier above, or the one after the
  // second pass, already saw every wave's last ring read.)
  MainTile& slot_w = wave == 0 ? ring0 : wave == 1 ? ring1 : wave == 2 ? ring2 : ring3;
  uint16_t* const stage = reinterpret_cast<uint16_t*>(&slot_w);
  const int64_t row0 = (int64_t)qb * kQPerWG + wave * kQPerWave;
  const int ch = lane & 7;
  constexpr int kRowSets = kQPerWave / 8;
  JoinArgs join{};
  uint64_t join_row0 = 0;
  uint32_t frame_rows = 0;
  // Token n is row n % P of frame n / P; a frame is H * P rows, of which this
  // head's start at join_row0 in frame 0.
  auto join_row = [&](int64_t row) {
    const uint32_t s = (uint32_t)row / (uint32_t)join.P;
    return join_row0 + (uint64_t)s * frame_rows + ((uint32_t)row - s * (uint32_t)join.P);
  };
  if constexpr (JOIN) {
    // Read from the argument segment only here (the empty asm keeps the loads
    // below the loop: held from the start they spill 9 SGPRs).
    typedef __attribute__((address_space(4))) const AttnJoinArgs* Args;
    Args args = (Args)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    join.o = args->join.o;
    join.lse = args->join.lse;
    join.P = args->join.P;
    const uint32_t heads = (uint32_t)args->a.H, jb = (uint32_t)bh / heads, jh = (uint32_t)bh % heads;
    frame_rows = heads * (uint32_t)join.P;
    join_row0 = ((uint64_t)jb * ((uint32_t)p.M / (uint32_t)join.P) * heads + jh) * (uint32_t)join.P;
    // The other attention's rows take the way of the stores below backwards:
    // whole rows into the stage, from where each lane reads the features of
    // its query where it will write the joined ones.
    u32x4 other[kRowSets];
#pragma unroll
    for (int i = 0; i < kRowSets; ++i) {
      const int64_t row = row0 + 8 * i + (lane >> 3);
      other[i] = row < p.M ? *reinterpret_cast<const u32x4*>(join.o + join_row(row) * kHD + ch * 8)
                           : u32x4{};
    }
#pragma unroll
    for (int i = 0; i < kRowSets; ++i) {
      const int r = 8 * i + (lane >> 3);
      *reinterpret_cast<u32x4*>(&stage[r * kHD + ((ch ^ (r & 7)) << 3)]) = other[i];
    }
  }
#pragma unroll
  for (int j = 0; j < kBlk; ++j) {
    const int r = 32 * j + l32;
    const int64_t row = q_base + 32 * j;
    const float l_tot = sum_halves(l_acc[j][0]);
    float inv = 1.0f / l_tot, w_other = 0.f;
    if constexpr (JOIN) {
      // Both halves in fp32; weights 2^(lse - max) over their sum.
      const float la = row < p.M ? join.lse[join_row(row)] : 0.f;
      const float lb = m_off[j] + __log2f(l_tot), top = fmaxf(la, lb);
      const float wa = __builtin_amdgcn_exp2f(la - top), wb = __builtin_amdgcn_exp2f(lb - top);
      const float norm = 1.0f / (wa + wb);
      w_other = wa * norm;
      inv *= wb * norm;
    }
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int cw = db * 4 + g;
        bf16x4* const at =
            reinterpret_cast<bf16x4*>(&stage[r * kHD + ((cw ^ (r & 7)) << 3) + 4 * hi]);
        bf16x4 ov;
        if constexpr (JOIN) {
          const bf16x4 x = *at;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            ov[e] = f32_to_half<F16>(__builtin_fmaf(half_to_f32<F16>(x[e]), w_other,
                                                    o_acc[j][db][4 * g + e] * inv));
        } else {
          ov = bf16x4{f32_to_half<F16>(o_acc[j][db][4 * g + 0] * inv),
                      f32_to_half<F16>(o_acc[j][db][4 * g + 1] * inv),
                      f32_to_half<F16>(o_acc[j][db][4 * g + 2] * inv),
                      f32_to_half<F16>(o_acc[j][db][4 * g + 3] * inv)};
        }
        *at = ov;
      }
    if (!JOIN && LSE && hi == 0 && row < p.M) LSE[row] = m_off[j] + __log2f(l_tot);
  }
  // All eight row reads first, then the stores (read-wait-store in turn
  // serialised eight LDS round trips).
  u32x4 ov16[kRowSets];
#pragma unroll
  for (int i = 0; i < kRowSets; ++i) {
    const int r = 8 * i + (lane >> 3);
    ov16[i] = *reinterpret_cast<const u32x4*>(&stage[r * kHD + ((ch ^ (r & 7)) << 3)]);
  }
  if (p.o16) {
#pragma unroll
    for (int i = 0; i < kRowSets; ++i) {
      const int64_t row = row0 + 8 * i + (lane >> 3);
      if (row < p.M) *reinterpret_cast<u32x4*>(O + row * o_sm + ch * 8) = ov16[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < kRowSets; ++i) {
      const int64_t row = row0 + 8 * i + (lane >> 3);
      if (row < p.M) {
        u32x2* dst = reinterpret_cast<u32x2*>(O + row * o_sm + ch * 8);
        dst[0] = u32x2{ov16[i][0], ov16[i][1]};
        dst[1] = u32x2{ov16[i][2], ov16[i][3]};
      }
    }
  }
}

template <bool F16>
__global__ __launch_bounds__(kThreads, 2) void attn_main_kernel(AttnArgs p) {
  attn_main_body<F16, false, false>(p);
}

// bf16 attention without bias (the frame and own-frame attentions): one launch
// where filling the records was another.  16 heads, 1,374 queries and keys per
// frame: 1 frame 29.0 -> 27.0 us, 4 frames 45.4 -> 43.1, 16 frames 135.5 ->
// 131.6, 100 frames (own keys) 854 -> 845.
__global__ __launch_bounds__(kThreads, 2) void attn_plain_kernel(AttnArgs p) {
  attn_main_body<false, false, true>(p);
}

// The second attention of a split key set, joined with the first in its
// epilogue: one read of the first's rows instead of writing this one's,
// reading both back and another launch (26 us at 16 frames, 21,984 queries,
// 16 heads; with the shared set written by one kernel too, the block went
// from 569 to 524 us).
template <bool F16>
__global__ __launch_bounds__(kThreads, 2) void attn_join_kernel(AttnJoinArgs p) {
  attn_main_body<F16, true, false>(p.a);
}

// Workspace: one row of ntiles tile records per (batch, head), then
// kBoundWords floats of row bounds per (batch, head), then one flag byte per
// wave.
size_t rec_bytes(int64_t B, int64_t H, int64_t N) {
  const int64_t ntiles = (N + kKT - 1) / kKT;
  return (size_t)(B * H * ntiles) * kRec * sizeof(float);
}
size_t bounds_bytes(int64_t B, int64_t H) { return (size_t)(B * H) * kBoundWords * sizeof(float); }
size_t attn_ws_bytes(int64_t B, int64_t H, int64_t M, int64_t N) {
  const int64_t gx = (M + kQPerWG - 1) / kQPerWG;
  return rec_bytes(B, H, N) + bounds_bytes(B, H) + (size_t)(B * H * gx) * kWaves;
}

}  // namespace
}  // namespace gpa

using namespace gpa;

extern "C" size_t gpa_attn_keybias_workspace_bytes(int64_t B, int64_t H, int64_t M, int64_t N) {
  if (B <= 0 || H <= 0 || M <= 0 || N <= 0) return 0;
  return attn_ws_bytes(B, H, M, N);
}

namespace {

// Shared by the bf16 and fp16 entry points; `fn` names the entry point in
// error messages.
template <bool F16>
int attn_keybias_run(const char* fn, const void* q, const void* k, const void* v,
                     const void* bias, int bias_kind, int64_t bias_sb, int64_t bias_sh,
                     int64_t bias_sn, void* o, float* lse, int64_t B, int64_t H, int64_t M,
                     int64_t N, int64_t D, int64_t q_sb, int64_t q_sh, int64_t q_sm, int64_t k_sb,
                     int64_t k_sh, int64_t k_sn, int64_t v_sb, int64_t v_sh, int64_t v_sn,
                     int64_t o_sb, int64_t o_sh, int64_t o_sm, int64_t lse_sb, int64_t lse_sh,
                     void* workspace, size_t workspace_bytes, float sm_scale, void* stream,
                     const JoinArgs* join = nullptr) {
  gpa_clear_error();
  if (B < 0 || H < 0 || M < 0 || N < 0 || D < 0) {
    gpa_set_error("%s: negative size", fn);
    return GPA_E_INVALID;
  }
  if (B == 0 || H == 0 || M == 0) return GPA_OK;
  if (N == 0) {
    gpa_set_error("%s: empty key set (N=0)", fn);
    return GPA_E_INVALID;
  }
  if (D != kHD && !attn_any_dim_supported(D)) {
    gpa_set_error("%s: head_dim %lld unsupported (16, 32, 64, 128 or 256)", fn, (long long)D);
    return GPA_E_UNSUPPORTED;
  }
  if (!q || !k || !v || !o || (join && (!join->o || !join->lse))) {
    gpa_set_error("%s: null tensor pointer", fn);
    return GPA_E_INVALID;
  }
  if (join && (D != kHD || join->P <= 0 || M % join->P != 0 || M > 0x7fffffff ||
               H * join->P > 0x7fffffff || (uintptr_t)join->o % 16)) {
    gpa_set_error("%s: the joined attention takes head dim 64, M=%lld a multiple of P=%d and "
                  "16-byte aligned rows", fn, (long long)M, join->P);
    return GPA_E_INVALID;
  }
  if (bias_kind != GPA_BIAS_NONE && bias_kind != GPA_BIAS_F32 && bias_kind != GPA_BIAS_BF16 &&
      bias_kind != GPA_BIAS_F16) {
    gpa_set_error("%s: unknown bias kind %d", fn, bias_kind);
    return GPA_E_INVALID;
  }
  if (bias_kind != GPA_BIAS_NONE && !bias) {
    gpa_set_error("%s: bias kind %d with a null bias pointer", fn, bias_kind);
    return GPA_E_INVALID;
  }
  if (!(sm_scale > 0.f) || !isfinite(sm_scale)) {
    gpa_set_error("%s: sm_scale must be positive and finite", fn);
    return GPA_E_INVALID;
  }
  const bool aligned = ((uintptr_t)q % 16 == 0) && ((uintptr_t)k % 16 == 0) &&
                       ((uintptr_t)v % 16 == 0) && ((uintptr_t)o % 8 == 0) && q_sm % 8 == 0 &&
                       q_sb % 8 == 0 && q_sh % 8 == 0 && k_sn % 8 == 0 && k_sb % 8 == 0 &&
                       k_sh % 8 == 0 && v_sn % 8 == 0 && v_sb % 8 == 0 && v_sh % 8 == 0 &&
                       o_sm % 4 == 0 && o_sb % 4 == 0 && o_sh % 4 == 0;
  if (!aligned || q_sm < D || k_sn < D || v_sn < D || o_sm < D) {
    gpa_set_error("%s: rows must have unit feature stride, q/k/v rows "
                  "16-byte and o rows 8-byte aligned", fn);
    return GPA_E_INVALID;
  }
  if (o_sm > 0x7fffffffLL) {
    gpa_set_error("%s: output row stride %lld exceeds 2^31 elements", fn, (long long)o_sm);
    return GPA_E_UNSUPPORTED;
  }
  if (B * H > 65535) {
    gpa_set_error("%s: B*H=%lld exceeds the grid limit", fn, (long long)(B * H));
    return GPA_E_UNSUPPORTED;
  }
  const int64_t gx = (M + kQPerWG - 1) / kQPerWG;
  if (gx * B * H > 0xffffffffLL) {   // the main pass numbers its workgroups in 32 bits
    gpa_set_error("%s: %lld query blocks exceed the grid limit", fn, (long long)(gx * B * H));
    return GPA_E_UNSUPPORTED;
  }
  // Buffer offsets are 32-bit: one (batch, head) slice of K and V, plus the
  // tiles fetched past its end, must stay below 2^31 bytes.
  const int64_t span = N + (kMainAhead + 1) * kKT;
  if (gx > 0x7fffffff || span * k_sn * 2 >= ((int64_t)1 << 31) ||
      span * v_sn * 2 >= ((int64_t)1 << 31)) {
    gpa_set_error("%s: one head's K/V slice exceeds 2 GiB", fn);
    return GPA_E_UNSUPPORTED;
  }
  const size_t ws_need = attn_ws_bytes(B, H, M, N);
  if (!workspace || workspace_bytes < ws_need || (uintptr_t)workspace % 16) {
    gpa_set_error("%s: 16-byte aligned workspace of %zu bytes required, %zu "
                  "given", fn,
                  ws_need, workspace ? workspace_bytes : (size_t)0);
    return GPA_E_WORKSPACE;
  }
  hipStream_t s = (hipStream_t)stream;
  const int64_t ntiles = (N + kKT - 1) / kKT;
  const float c = sm_scale * kLog2e;
  if (D != kHD) {
    // Head dims other than 64 (attn_any_dim.hip): their bias rows (4 bytes
    // per key) fit in the records' place (144 bytes per 32 keys).
    if (((M + 127) / 128) * B * H > 0xffffffffLL) {   // 128-query workgroups, 32-bit numbering
      gpa_set_error("%s: %lld query blocks exceed the grid limit", fn,
                    (long long)(((M + 127) / 128) * B * H));
      return GPA_E_UNSUPPORTED;
    }
    if (attn_any_dim_ws_bytes(B * H, N) > rec_bytes(B, H, N)) {
      gpa_set_error("%s: internal: bias rows exceed the workspace", fn);
      return GPA_E_WORKSPACE;
    }
    AnyDimArgs g{};
    g.q = (const uint16_t*)q;
    g.k = (const uint16_t*)k;
    g.v = (const uint16_t*)v;
    g.bias = bias;
    g.o = (uint16_t*)o;
    g.lse = lse;
    g.H = (int)H;
    g.BH = B * H;
    g.M = M;
    g.N = N;
    g.q_sb = q_sb; g.q_sh = q_sh; g.q_sm = q_sm;
    g.k_sb = k_sb; g.k_sh = k_sh; g.k_sn = k_sn;
    g.v_sb = v_sb; g.v_sh = v_sh; g.v_sn = v_sn;
    g.o_sb = o_sb; g.o_sh = o_sh; g.o_sm = o_sm;
    g.bias_sb = bias_sb; g.bias_sh = bias_sh; g.bias_sn = bias_sn;
    g.lse_sb = lse_sb; g.lse_sh = lse_sh;
    g.c = c;
    g.mul = 1.0f / sm_scale;
    g.ws = (float*)workspace;
    g.ws_bytes = workspace_bytes;
    const hipError_t ge = attn_any_dim_launch<F16>(g, D, bias_kind, s);
    if (ge != hipSuccess) {
      gpa_set_error("%s: launch failed: %s", fn, hipGetErrorString(ge));
      return GPA_E_LAUNCH;
    }
    return GPA_OK;
  }

  RecArgs ra{};
  ra.k = (const uint16_t*)k;
  ra.bias = bias;
  ra.recs = (float*)workspace;
  ra.H = (int)H;
  ra.k_sb = k_sb; ra.k_sh = k_sh; ra.k_sn = k_sn;
  ra.sb = bias_sb; ra.sh = bias_sh; ra.sn = bias_sn;
  ra.N = N;
  ra.ntiles = ntiles;
  if (B * H * ntiles > 0x7fffffff) {
    gpa_set_error("%s: %lld key tiles exceed the grid limit", fn, (long long)(B * H * ntiles));
    return GPA_E_UNSUPPORTED;
  }
  ra.mul = 1.0f / sm_scale;
  ra.c = c;
  ra.total = B * H * ntiles;
  float* bounds = (float*)((char*)workspace + rec_bytes(B, H, N));
  const bool no_bound = bias_kind == GPA_BIAS_NONE && !F16;
  const bool plain = no_bound && !join;
  if (plain) {
  } else if (no_bound) {
    const int64_t n = ra.total * kRec;
    hipLaunchKernelGGL(fill_records_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                       (float*)workspace, bounds, ntiles, N, ra.total, B * H);
  } else {
    const dim3 rgrid((unsigned)((ra.total + kRecTiles - 1) / kRecTiles)), rblock(256);
    switch (bias_kind) {
      case GPA_BIAS_F32:
        hipLaunchKernelGGL((tile_records_kernel<F16, GPA_BIAS_F32>), rgrid, rblock, 0, s, ra);
        break;
      case GPA_BIAS_BF16:
        hipLaunchKernelGGL((tile_records_kernel<F16, GPA_BIAS_BF16>), rgrid, rblock, 0, s, ra);
        break;
      case GPA_BIAS_F16:
        hipLaunchKernelGGL((tile_records_kernel<F16, GPA_BIAS_F16>), rgrid, rblock, 0, s, ra);
        break;
      default:
        hipLaunchKernelGGL((tile_records_kernel<F16, GPA_BIAS_NONE>), rgrid, rblock, 0, s, ra);
        break;
    }
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    gpa_set_error("%s: tile-record pre-pass launch failed: %s", fn,
                  hipGetErrorString(e));
    return GPA_E_LAUNCH;
  }
  const bool fold = !no_bound && ntiles <= kFoldTiles && gx * B * H <= kFoldGrid;
  if (!no_bound && !fold) {
    hipLaunchKernelGGL(row_bounds_kernel, dim3((unsigned)(B * H)), dim3(256), 0, s,
                       (const float*)workspace, bounds, ntiles);
    e = hipGetLastError();
    if (e != hipSuccess) {
      gpa_set_error("%s: row-bound pre-pass launch failed: %s", fn,
                    hipGetErrorString(e));
      return GPA_E_LAUNCH;
    }
  }

  AttnArgs p{};
  p.q = (const uint16_t*)q;
  p.k = (const uint16_t*)k;
  p.v = (const uint16_t*)v;
  p.recs = (const float*)workspace;
  p.bounds = bounds;
  p.flags = (uint8_t*)bounds + bounds_bytes(B, H);
  p.o = (uint16_t*)o;
  p.lse = lse;
  p.H = (int)H;
  p.M = M;
  p.N = N;
  p.q_sb = q_sb; p.q_sh = q_sh; p.q_sm = q_sm;
  p.k_sb = k_sb; p.k_sh = k_sh; p.k_sn = k_sn;
  p.v_sb = v_sb; p.v_sh = v_sh; p.v_sn = v_sn;
  p.o_sb = o_sb; p.o_sh = o_sh; p.o_sm = o_sm;
  p.lse_sb = lse_sb; p.lse_sh = lse_sh;
  p.k_bytes = (uint32_t)(((N - 1) * k_sn + D) * 2);
  p.v_bytes = (uint32_t)(((N - 1) * v_sn + D) * 2);
  p.rec_bytes = (uint32_t)(ntiles * kRec * sizeof(float));
  p.c = c;
  p.o16 = ((uintptr_t)o % 16 == 0 && o_sm % 8 == 0 && o_sb % 8 == 0 && o_sh % 8 == 0) ? 1 : 0;
  p.no_bound = no_bound ? 1 : 0;
  p.fold = fold ? 1 : 0;

  const dim3 grid((unsigned)gx, (unsigned)(B * H)), block(kThreads);
  if (join)
    hipLaunchKernelGGL(attn_join_kernel<F16>, grid, block, 0, s, AttnJoinArgs{p, *join});
  else if (plain)
    hipLaunchKernelGGL(attn_plain_kernel, grid, block, 0, s, p);
  else
    hipLaunchKernelGGL(attn_main_kernel<F16>, grid, block, 0, s, p);
  e = hipGetLastError();
  if (e != hipSuccess) {
    gpa_set_error("%s: launch failed: %s", fn, hipGetErrorString(e));
    return GPA_E_LAUNCH;
  }
  return GPA_OK;
}

}  // namespace

extern "C" int gpa_attn_keybias_bf16(const void* q, const void* k, const void* v, const void* bias,
                                     int bias_kind, int64_t bias_sb, int64_t bias_sh,
                                     int64_t bias_sn, void* o, float* lse, int64_t B, int64_t H,
                                     int64_t M, int64_t N, int64_t D, int64_t q_sb, int64_t q_sh,
                                     int64_t q_sm, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                                     int64_t v_sb, int64_t v_sh, int64_t v_sn, int64_t o_sb,
                                     int64_t o_sh, int64_t o_sm, int64_t lse_sb, int64_t lse_sh,
                                     void* workspace, size_t workspace_bytes, float sm_scale,
                                     void* stream) {
  return attn_keybias_run<false>("gpa_attn_keybias_bf16", q, k, v, bias, bias_kind, bias_sb,
                                 bias_sh, bias_sn, o, lse, B, H, M, N, D, q_sb, q_sh, q_sm, k_sb,
                                 k_sh, k_sn, v_sb, v_sh, v_sn, o_sb, o_sh, o_sm, lse_sb, lse_sh,
                                 workspace, workspace_bytes, sm_scale, stream);
}

extern "C" int gpa_attn_keybias_f16(const void* q, const void* k, const void* v, const void* bias,
                                    int bias_kind, int64_t bias_sb, int64_t bias_sh,
                                    int64_t bias_sn, void* o, float* lse, int64_t B, int64_t H,
                                    int64_t M, int64_t N, int64_t D, int64_t q_sb, int64_t q_sh,
                                    int64_t q_sm, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                                    int64_t v_sb, int64_t v_sh, int64_t v_sn, int64_t o_sb,
                                    int64_t o_sh, int64_t o_sm, int64_t lse_sb, int64_t lse_sh,
                                    void* workspace, size_t workspace_bytes, float sm_scale,
                                    void* stream) {
  return attn_keybias_run<true>("gpa_attn_keybias_f16", q, k, v, bias, bias_kind, bias_sb,
                                bias_sh, bias_sn, o, lse, B, H, M, N, D, q_sb, q_sh, q_sm, k_sb,
                                k_sh, k_sn, v_sb, v_sh, v_sn, o_sb, o_sh, o_sm, lse_sb, lse_sh,
                                workspace, workspace_bytes, sm_scale, stream);
}

extern "C" int gpa_attn_keybias_join(
    int dtype, const void* q, const void* k, const void* v, const void* bias, int bias_kind,
    int64_t bias_sb, int64_t bias_sh, int64_t bias_sn, const void* other_o, const float* other_lse,
    int64_t P, void* o, int64_t B, int64_t H, int64_t M, int64_t N, int64_t D, int64_t q_sb, int64_t q_sh, int64_t q_sm, int64_t k_sb, int64_t k_sh,
    int64_t k_sn, int64_t v_sb, int64_t v_sh, int64_t v_sn, int64_t o_sb, int64_t o_sh,
    int64_t o_sm, void* workspace, size_t workspace_bytes, float sm_scale, void* stream) {
  static const char* fn = "gpa_attn_keybias_join";
  const JoinArgs join{(const uint16_t*)other_o, other_lse, P > 0 && P <= 0x7fffffff ? (int)P : 0};
  if (dtype == GPA_DTYPE_BF16)
    return attn_keybias_run<false>(fn, q, k, v, bias, bias_kind, bias_sb, bias_sh, bias_sn, o,
                                   nullptr, B, H, M, N, D, q_sb, q_sh, q_sm, k_sb, k_sh, k_sn,
                                   v_sb, v_sh, v_sn, o_sb, o_sh, o_sm, 0, 0, workspace,
                                   workspace_bytes, sm_scale, stream, &join);
  if (dtype == GPA_DTYPE_F16)
    return attn_keybias_run<true>(fn, q, k, v, bias, bias_kind, bias_sb, bias_sh, bias_sn, o,
                                  nullptr, B, H, M, N, D, q_sb, q_sh, q_sm, k_sb, k_sh, k_sn,
                                  v_sb, v_sh, v_sn, o_sb, o_sh, o_sm, 0, 0, workspace,
                                  workspace_bytes, sm_scale, stream, &join);
  gpa_clear_error();
  gpa_set_error("%s: unknown dtype %d", fn, dtype);
  return GPA_E_INVALID;
}

// ---------------------------------------------------------------------------
// The allocation-free variant: the workspace is a device-resident array of
// this file.  Each GPU the library runs on holds its own copy (allocated by
// the runtime with the code object, kept until the process ends).  Host code
// never passes the array's name to a kernel: on the host that name is a
// stand-in, not a device address.  The device address is resolved once per
// device with hipGetSymbolAddress, on that device's first call, and every
// later use goes through the resolved pointer.
//
// The pre-passes and the main pass write every workspace byte a call reads
// (tile records, row bounds, one flag per wave) before reading it, so nothing
// has to be cleared between calls.  Calls that overlap on one GPU (two host
// threads, or two streams) share the array and race.
static __device__ __attribute__((aligned(256))) uint8_t scratch[GPA_ATTN_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxScratchDevices] = {};

// Device address of this GPU's `scratch` (the current device's), or nullptr
// with the error message set.
void* scratch_for_current_device(const char* fn) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    gpa_set_error("%s: hipGetDevice failed: %s", fn, hipGetErrorString(e));
    return nullptr;
  }
  if (dev < 0 || dev >= kMaxScratchDevices) {
    gpa_set_error("%s: device %d is beyond the %d devices the scratch table holds", fn, dev,
                  kMaxScratchDevices);
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      gpa_set_error("%s: hipGetSymbolAddress(scratch) failed on device %d: %s", fn, dev,
                    hipGetErrorString(e));
      return nullptr;
    }
    g_scratch_ptr[dev] = ptr;
  }
  return g_scratch_ptr[dev];
}

}  // namespace

extern "C" int gpa_attn_keybias_bf16_noalloc(
    const void* q, const void* k, const void* v, const void* bias, int bias_kind,
    int64_t bias_sb, int64_t bias_sh, int64_t bias_sn, void* o, float* lse, int64_t B, int64_t H,
    int64_t M, int64_t N, int64_t D, int64_t q_sb, int64_t q_sh, int64_t q_sm, int64_t k_sb,
    int64_t k_sh, int64_t k_sn, int64_t v_sb, int64_t v_sh, int64_t v_sn, int64_t o_sb,
    int64_t o_sh, int64_t o_sm, int64_t lse_sb, int64_t lse_sh, float sm_scale, void* stream) {
  static const char* fn = "gpa_attn_keybias_bf16_noalloc";
  gpa_clear_error();
  if (B > 0 && H > 0 && M > 0 && N > 0) {
    const size_t need = attn_ws_bytes(B, H, M, N);
    if (need > (size_t)GPA_ATTN_NOALLOC_SCRATCH_BYTES) {
      gpa_set_error("%s: this shape needs %zu bytes of workspace, the static scratch holds %zu "
                    "(use gpa_attn_keybias_bf16 with a caller workspace)",
                    fn, need, (size_t)GPA_ATTN_NOALLOC_SCRATCH_BYTES);
      return GPA_E_UNSUPPORTED;
    }
  }
  void* ws = scratch_for_current_device(fn);
  if (!ws) return GPA_E_LAUNCH;
  return attn_keybias_run<false>(fn, q, k, v, bias, bias_kind, bias_sb, bias_sh, bias_sn, o, lse,
                                 B, H, M, N, D, q_sb, q_sh, q_sm, k_sb, k_sh, k_sn, v_sb, v_sh,
                                 v_sn, o_sb, o_sh, o_sm, lse_sb, lse_sh, ws,
                                 (size_t)GPA_ATTN_NOALLOC_SCRATCH_BYTES, sm_scale, stream);
}
