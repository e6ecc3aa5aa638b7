// Biased flash attention for head dims other than 64 (16, 32, 128, 256):
// the same contract as attn_main_kernel (scores q.k * sm_scale + bias in the
// exp2 domain, fp32 online softmax, P rounded to the operand format for the
// P.V product, fp32 accumulation, log2 LSE).  The reference kernel takes
// HEAD_DIM as a constexpr (merging/fused_attention.py:82, 89, 97) and its
// wrapper reads it from q (:146, 177); VGGT uses 64, which the main kernel
// serves.  Row sums add the fp32 P, as the reference's do (:113).
//
// Common to the tiled and the narrow kernel below
//   * Scores are computed transposed, S^T = K . Q^T, on v_mfma_f32_32x32x16
//     (HD / 16 k-steps): a lane owns one query of a 32-query block and 16 of
//     the tile's 32 keys (the other 16 sit in lane^32); the accumulator
//     starts from the keys' bias / sm_scale (-inf past N), and P^T is used in
//     place as the B operand of O^T = V^T . P^T.
//   * The bias comes from a pre-pass (bias_rows_kernel): per (batch, head)
//     one fp32 row of bias / sm_scale over the keys rounded up to whole
//     tiles, -inf past N, in the workspace.
//   * K, V and the bias stream through a four-slot LDS ring of 32-key tiles
//     filled by buffer_load ... lds (DMA, no staging registers), three tiles
//     ahead; rows past N read zeros by range.
//   * Software pipelining by one tile: iteration t computes S(t+1) on the
//     matrix pipe beside the softmax of S(t) on the VALU, then O += V(t)^T .
//     P(t)^T.
//   * Workgroups are renumbered XCD-aware so the query blocks of one (batch,
//     head) share an XCD's L2 for their K/V stream.
#include "gpa_common.h"

#include <math.h>

#include "attn_any_dim.h"

namespace gpa {
namespace {

constexpr int kAWaves = 4;
constexpr int kAThreads = kAWaves * 64;
constexpr int kAQ = kAWaves * 32;            // queries per workgroup (tiled and short kernels)
constexpr int kAKT = 32;                      // keys per tile

template <int KIND>
__device__ __forceinline__ float any_bias(const void* bias, int64_t off) {
  if constexpr (KIND == GPA_BIAS_F32) return static_cast<const float*>(bias)[off];
  else if constexpr (KIND == GPA_BIAS_BF16)
    return __uint_as_float((uint32_t)static_cast<const uint16_t*>(bias)[off] << 16);
  else if constexpr (KIND == GPA_BIAS_F16)
    return (float)__builtin_bit_cast(_Float16, static_cast<const uint16_t*>(bias)[off]);
  else return 0.f;
}

// ---------------------------------------------------------------------------
// Head dims 128 and 256: the tiled kernel.
//
// One 32-query block per wave (128 queries per workgroup):
//   * A lazily moved offset: m starts at tile 0's exact row max and moves to
//     a tile's row max only when that exceeds m + kLazyUp (64 log2 units for
//     bf16 P, which has fp32's exponent range; 15 for fp16 P, below 65504),
//     in a wave-uniform branch.  Every P stays <= 2^kLazyUp and each row's
//     largest P >= 1, the row sums (fp32, of the fp32 P, as the reference)
//     and O stay far inside fp32, and the softmax is the same; after the
//     first tiles of a row the branch is rarely taken.
//   * K rows are stored with their 16-byte chunks XOR-swizzled by key & 15
//     (a 16-lane pass of fragment reads hits 16 distinct chunks), V rows
//     row-major with chunks swizzled by (key & 3) << 2, and the V^T operand
//     is read with ds_read_b64_tr_b16 (a 32-lane pass covers all 64 banks
//     once).  The DMA lanes pick the global chunk their LDS position holds,
//     so the swizzle costs nothing.
// Two blocks per wave would halve the LDS reads per MFMA, but at 128 their
// registers leave one wave per SIMD: 787 against 686 us at 16 heads, 16,488
// queries and 4,993 keys.

template <bool F16> constexpr float kLazyUp = F16 ? 15.0f : 64.0f;
constexpr int kLSlots = 4;                    // ring slots: tiles t .. t+3

template <int KIND>
__global__ __launch_bounds__(256) void bias_rows_kernel(const void* bias, float* rows, int H,
                                                        int64_t N, int64_t npad, int64_t sb,
                                                        int64_t sh, int64_t sn, float mul) {
  const int64_t bh = blockIdx.y;
  const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (n >= npad) return;
  float x = -INFINITY;
  if (n < N) {
    if constexpr (KIND == GPA_BIAS_NONE) x = 0.f;
    else x = any_bias<KIND>(bias, (bh / H) * sb + (bh % H) * sh + n * sn) * mul;
  }
  rows[bh * npad + n] = x;
}

// DMA of 4 / 16 bytes per lane into LDS at lds + 4 * lane / lds + 16 * lane.
__device__ __forceinline__ void lds_dma4(__amdgpu_buffer_rsrc_t r, void* lds, uint32_t voff,
                                         uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      r, (__attribute__((address_space(3))) void*)lds, 4, voff, soff, 0, 0);
}
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t r, void* lds, uint32_t voff,
                                          uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      r, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, 0, 0);
}
// Wait until at most N vector-memory instructions of this wave are in flight.
template <int N>
__device__ __forceinline__ void wait_vmem() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// One ring slot: a tile's K and V rows (swizzled as above) and its bias
// words (64 words: the DMA of one wave writes 4 bytes per lane).
template <int HD>
struct TiledSlot {
  uint16_t k[kAKT * HD];
  uint16_t v[kAKT * HD];
  float b[64];
};

template <int HD, bool F16>
__global__ __launch_bounds__(kAThreads, HD >= 256 ? 1 : 2) void attn_tiled_kernel(AnyDimArgs p) {
  constexpr int KS = HD / 16;                 // k-steps of the score product
  constexpr int DB = HD / 32;                 // 32-feature blocks of O
  constexpr int CH = HD / 8;                  // 16-byte chunks per key row
  constexpr int DJ = kAKT * CH / kAThreads;   // 16-byte DMAs per wave, tile and tensor
  constexpr int OPS = 2 * DJ + 1;             // DMA instructions per wave and tile
  static_assert(kAKT * CH % kAThreads == 0, "whole DMA instructions per wave");
  static_assert(kLSlots == 4, "the loop below is unrolled over four slots");
  // Four statically named slots: the compiler then knows which in-flight DMA
  // each LDS read may depend on (with one array and a runtime slot index it
  // waits for every DMA before every read).
  __shared__ __attribute__((aligned(16))) TiledSlot<HD> r0, r1, r2, r3;
  __shared__ __attribute__((aligned(16))) float b_sink[64];

  const int tid = threadIdx.x, lane = tid & 63, hi = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int qb, bhi;
  {
    const uint32_t T = gridDim.x * gridDim.y, L = blockIdx.y * gridDim.x + blockIdx.x;
    const uint32_t q8 = T / 8, r8 = T % 8, x = L % 8;
    const uint32_t item = x * q8 + (x < r8 ? x : r8) + L / 8;
    qb = (int)(item % gridDim.x);
    bhi = (int)(item / gridDim.x);
  }
  const int64_t bh = bhi, b = bh / p.H, h = bh % p.H;
  const int64_t q_row = (int64_t)qb * kAQ + wave * 32 + l32;
  const uint16_t* Q = p.q + b * p.q_sb + h * p.q_sh;
  const uint16_t* K = p.k + b * p.k_sb + h * p.k_sh;
  const uint16_t* V = p.v + b * p.v_sb + h * p.v_sh;
  const int ntiles = (int)((p.N + kAKT - 1) / kAKT);
  const float* Brow = p.ws + bh * (int64_t)ntiles * kAKT;
  const float c = p.c;

  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    qf[ks] = q_row < p.M ? *reinterpret_cast<const bf16x8*>(Q + q_row * p.q_sm + 16 * ks + 8 * hi)
                         : bf16x8{};
  __builtin_amdgcn_sched_barrier(0);

  const uint32_t k_row = (uint32_t)p.k_sn * 2u, v_row = (uint32_t)p.v_sn * 2u;
  const __amdgpu_buffer_rsrc_t krs = make_rsrc(K, (uint32_t)((p.N - 1) * p.k_sn * 2 + HD * 2));
  const __amdgpu_buffer_rsrc_t vrs = make_rsrc(V, (uint32_t)((p.N - 1) * p.v_sn * 2 + HD * 2));
  const __amdgpu_buffer_rsrc_t brs = make_rsrc(Brow, (uint32_t)ntiles * kAKT * 4u);
  // LDS chunk position (wave DJ + j) 64 + lane holds key pos / CH, physical
  // chunk pos % CH, i.e. the logical chunk that the XOR swizzle maps there.
  uint32_t k_voff[DJ], v_voff[DJ];
#pragma unroll
  for (int j = 0; j < DJ; ++j) {
    const int pos = (wave * DJ + j) * 64 + lane;
    const int key = pos / CH, pch = pos % CH;
    k_voff[j] = key * k_row + (uint32_t)((pch ^ (key & 15)) * 16);
    v_voff[j] = key * v_row + (uint32_t)((pch ^ ((key & 3) << 2)) * 16);
  }
  // Wave 0's first 32 lanes fetch the tile's 32 bias words; the other lanes
  // point past the descriptor's range and land zeros (waves 1-3 into a sink,
  // so that every wave issues the same DMAs and waits).
  const uint32_t b_voff = (wave == 0 && lane < kAKT) ? (uint32_t)lane * 4u : 0x40000000u;
  auto issue = [&](int t, TiledSlot<HD>& S) {
    const uint32_t n0 = (uint32_t)t * kAKT;
#pragma unroll
    for (int j = 0; j < DJ; ++j) lds_dma16(krs, &S.k[(wave * DJ + j) * 512], k_voff[j], n0 * k_row);
#pragma unroll
    for (int j = 0; j < DJ; ++j) lds_dma16(vrs, &S.v[(wave * DJ + j) * 512], v_voff[j], n0 * v_row);
    float* dst = wave == 0 ? &S.b[0] : &b_sink[0];
    lds_dma4(brs, dst, b_voff, n0 * 4u);
  };

  int k_off[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) k_off[ks] = l32 * HD + (((2 * ks + hi) ^ (l32 & 15)) << 3);
  // V^T operand: lane (hi, bit 4, v = (lane & 15) >> 2, a = lane & 3) points
  // at key 4 hi + v (+ 16 s + 8 e), features 32 db + 16 bit4 + 4 a .. +3;
  // ds_read_b64_tr_b16 then hands lane l feature 32 db + l % 32 of keys
  // 16 s + 8 e + 4 hi .. +3, the key order of the score MFMA's registers.
  int v_off[DB];
  {
    const int v4 = (lane & 15) >> 2, a = lane & 3, bit4 = (lane >> 4) & 1;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int lc = 4 * db + 2 * bit4 + (a >> 1);
      v_off[db] = (4 * hi + v4) * HD + ((lc ^ (v4 << 2)) << 3) + (a & 1) * 4;
    }
  }

  auto scores = [&](const TiledSlot<HD>& S) {
    f32x16 sv;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 bv = *reinterpret_cast<const f32x4*>(&S.b[8 * g + 4 * hi]);
      sv[4 * g + 0] = bv[0];
      sv[4 * g + 1] = bv[1];
      sv[4 * g + 2] = bv[2];
      sv[4 * g + 3] = bv[3];
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const bf16x8 kf = *reinterpret_cast<const bf16x8*>(&S.k[k_off[ks]]);
      sv = mfma32x32x16_t<F16>(kf, qf[ks], sv);
    }
    return sv;
  };
  auto row_max = [&](const f32x16& x) {
    float mx = fmaxf(fmaxf(x[0], x[1]), x[2]);
#pragma unroll
    for (int r = 3; r < 15; r += 2) mx = fmaxf(fmaxf(mx, x[r]), x[r + 1]);
    mx = fmaxf(mx, x[15]);
    return max_halves(mx) * c;
  };

  f32x16 o_acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o_acc[db] = f32x16{};
  float l = 0.f;

  issue(0, r0);
  issue(1, r1);
  issue(2, r2);
  wait_vmem<2 * OPS>();
  __syncthreads();
  f32x16 s_cur = scores(r0);
  float m = fmaxf(row_max(s_cur), -1.0e30f);  // finite: a tile of -inf biases scores 0

  // Iteration t: tile t in `cur`, tile t+1 in `nxt`, tile t+3 issued into
  // `dst` (the slot of tile t-1, free once every wave passed the barrier).
  auto iter = [&](int t, const TiledSlot<HD>& cur, const TiledSlot<HD>& nxt,
                  TiledSlot<HD>& dst) {
    wait_vmem<OPS>();                         // tile t+1 landed (tile t+2 in flight)
    __syncthreads();                          // ... for every wave
    issue(t + 3, dst);
    const f32x16 s_nxt = scores(nxt);
    // The V^T fragments of tile t, all read before the softmax (read after
    // it, their LDS latency sat between the softmax and the P.V product:
    // head dim 256 45.2 -> 35.6 ms, 128 32.5 -> 31.5 ms, same box).
    bf16x8 vf[DB][2];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        typedef short i16x4 __attribute__((ext_vector_type(4)));
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) i16x4*)&cur.v[v_off[db] + 16 * s * HD]);
        const i16x4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) i16x4*)&cur.v[v_off[db] + (16 * s + 8) * HD]);
        const bf16x4 l4 = __builtin_bit_cast(bf16x4, lo), u4 = __builtin_bit_cast(bf16x4, up);
        vf[db][s] = bf16x8{l4[0], l4[1], l4[2], l4[3], u4[0], u4[1], u4[2], u4[3]};
      }
    // Softmax of S(t): move the offset only where the row max left the window.
    const float mx = row_max(s_cur);
    const bool move = mx > m + kLazyUp<F16>;
    if (__builtin_amdgcn_ballot_w64(move)) {
      const float m_new = move ? mx : m;
      const float alpha = __builtin_amdgcn_exp2f(m - m_new);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db) o_acc[db] *= alpha;
    }
    bf16x8 pb[2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s_cur[8 * s + e], c, -m));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s_cur[8 * s + e + 1], c, -m));
        l += p0 + p1;
        const bf16x2 pv2 = pack2<F16>(p0, p1);
        pb[s][e] = pv2[0];
        pb[s][e + 1] = pv2[1];
      }
    // O^T += V^T . P^T
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int s = 0; s < 2; ++s) o_acc[db] = mfma32x32x16_t<F16>(vf[db][s], pb[s], o_acc[db]);
    s_cur = s_nxt;
  };
  for (int t = 0; t < ntiles; t += 4) {
    iter(t, r0, r1, r3);
    if (t + 1 >= ntiles) break;
    iter(t + 1, r1, r2, r0);
    if (t + 2 >= ntiles) break;
    iter(t + 2, r2, r3, r1);
    if (t + 3 >= ntiles) break;
    iter(t + 3, r3, r0, r2);
  }
  wait_vmem<0>();                             // no DMA may land after the workgroup ends

  const float l_tot = sum_halves(l);
  if (q_row >= p.M) return;
  const float inv = 1.0f / l_tot;
  uint16_t* O = p.o + b * p.o_sb + h * p.o_sh + q_row * p.o_sm;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int f0 = db * 32 + 8 * g + 4 * hi;
      const bf16x2 lo = pack2<F16>(o_acc[db][4 * g + 0] * inv, o_acc[db][4 * g + 1] * inv);
      const bf16x2 up = pack2<F16>(o_acc[db][4 * g + 2] * inv, o_acc[db][4 * g + 3] * inv);
      *reinterpret_cast<u32x2*>(O + f0) =
          u32x2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, up)};
    }
  if (p.lse && hi == 0) p.lse[b * p.lse_sb + h * p.lse_sh + q_row] = m + __log2f(l_tot);
}

// ---------------------------------------------------------------------------
// Head dims 16 and 32, few keys or a small grid: one 32-query block per wave.
//
// What bounds such a call is its launches and one workgroup's walk over the
// keys, not the chip.  So the bias is read where it lies (a pre-pass for it is
// another launch, 2.5 us), a wave carries one block of 32 queries (with two,
// half the waves do all the work of up to 128 queries), and the next tile's
// loads wait in registers while a tile is computed: a two-slot LDS ring, K
// row-major in padded rows, V transposed, each 16-key step's keys in the order
// the score MFMA's result registers enumerate them.  The offset is the running
// row max, O and the row sums rescaled on every tile.  At head dim 16 the P.V
// product runs on a 32-feature block whose upper 16 features are zero.
//
// Against the narrow kernel below, microseconds (32 bf16, bias; heads x
// queries, keys): 4 x 500, 64: 3.9 and 6.3; 16 x 1,374, 500: 12.7 and 15.6;
// 1,703: 37.8 and 37.8; 16 x 2,748, 500: 15.3 and 16.1; 1,000: 27.2 and 25.7;
// 128 x 1,374, 128: 12.7 and 13.4; 256: 21.0 and 19.6.

// Position of key k (0..31) of a tile in the transposed V rows: step s =
// k / 16 holds, in lane-half order, the keys the score MFMA's result
// registers 8s .. 8s+7 of lanes 0-31 (hi = 0) and 32-63 (hi = 1) hold:
// register r of half hi is key 8 (r / 4) + 4 hi + r % 4.
__device__ __forceinline__ int vt_pos(int k) {
  return (k & ~15) + ((k >> 2) & 1) * 8 + ((k >> 3) & 1) * 4 + (k & 3);
}

template <int HD, bool F16, int KIND>
__global__ __launch_bounds__(kAThreads, 2) void attn_short_kernel(AnyDimArgs p) {
  constexpr int KS = HD / 16;                 // k-steps of the score product
  constexpr int DB = HD >= 32 ? HD / 32 : 1;  // 32-feature blocks of O
  constexpr int KROW = HD + 8;                // padded K row (elements)
  constexpr int VROW = kAKT + 8;              // padded transposed V row
  constexpr int CH = HD / 8;                  // 16-byte chunks per key row
  constexpr int NCH = kAKT * CH;              // chunks per tile and tensor
  constexpr int CPT = (NCH + kAThreads - 1) / kAThreads;
  __shared__ __attribute__((aligned(16))) uint16_t ks_lds[2][kAKT * KROW];
  __shared__ __attribute__((aligned(16))) uint16_t vt_lds[2][DB * 32 * VROW];
  __shared__ __attribute__((aligned(16))) float bias_lds[2][kAKT];

  const int tid = threadIdx.x, lane = tid & 63, hi = lane >> 5, l32 = lane & 31;
  const int wave = tid >> 6;
  const int64_t bh = blockIdx.y, b = bh / p.H, h = bh % p.H;
  const int64_t q_row = (int64_t)blockIdx.x * kAQ + wave * 32 + l32;
  const uint16_t* Q = p.q + b * p.q_sb + h * p.q_sh;
  const uint16_t* K = p.k + b * p.k_sb + h * p.k_sh;
  const uint16_t* V = p.v + b * p.v_sb + h * p.v_sh;
  const int64_t boff = b * p.bias_sb + h * p.bias_sh;
  const float c = p.c;

  if constexpr (HD == 16) {                   // the zero upper half of the O block
    for (int i = tid; i < 2 * 32 * VROW; i += kAThreads) {
      const int sl = i / (32 * VROW), r = i % (32 * VROW);
      if (r >= 16 * VROW) vt_lds[sl][r] = 0;
    }
  }

  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    qf[ks] = q_row < p.M ? *reinterpret_cast<const bf16x8*>(Q + q_row * p.q_sm + 16 * ks + 8 * hi)
                         : bf16x8{};

  // One tile's K and V chunks and bias, into registers (zeros / -inf past N).
  u32x4 kreg[CPT], vreg[CPT];
  float breg = -INFINITY;
  auto load_tile = [&](int t) {
    const int64_t n0 = (int64_t)t * kAKT;
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int cidx = tid + i * kAThreads;
      const int key = cidx / CH, ch = cidx % CH;
      const bool ok = cidx < NCH && n0 + key < p.N;
      kreg[i] = ok ? *reinterpret_cast<const u32x4*>(K + (n0 + key) * p.k_sn + 8 * ch) : u32x4{};
      vreg[i] = ok ? *reinterpret_cast<const u32x4*>(V + (n0 + key) * p.v_sn + 8 * ch) : u32x4{};
    }
    if (tid < kAKT)
      breg = n0 + tid < p.N ? any_bias<KIND>(p.bias, boff + (n0 + tid) * p.bias_sn) * p.mul
                            : -INFINITY;
  };
  auto store_tile = [&](int sl) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int cidx = tid + i * kAThreads;
      if (cidx < NCH) {
        const int key = cidx / CH, ch = cidx % CH;
        *reinterpret_cast<u32x4*>(&ks_lds[sl][key * KROW + 8 * ch]) = kreg[i];
        const int pos = vt_pos(key);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          vt_lds[sl][(8 * ch + 2 * e) * VROW + pos] = (uint16_t)(vreg[i][e] & 0xffffu);
          vt_lds[sl][(8 * ch + 2 * e + 1) * VROW + pos] = (uint16_t)(vreg[i][e] >> 16);
        }
      }
    }
    if (tid < kAKT) bias_lds[sl][tid] = breg;
  };

  float m = -1.0e30f, l = 0.f;                // finite: a tile of -inf biases scores 0
  f32x16 o_acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o_acc[db] = f32x16{};

  const int ntiles = (int)((p.N + kAKT - 1) / kAKT);
  load_tile(0);
  store_tile(0);
  for (int t = 0; t < ntiles; ++t) {
    const int sl = t & 1;
    __syncthreads();                          // slot sl written; slot sl^1 free
    if (t + 1 < ntiles) load_tile(t + 1);
    // S^T = K . Q^T + bias / sm_scale
    f32x16 sv;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 bv = *reinterpret_cast<const f32x4*>(&bias_lds[sl][8 * g + 4 * hi]);
      sv[4 * g + 0] = bv[0];
      sv[4 * g + 1] = bv[1];
      sv[4 * g + 2] = bv[2];
      sv[4 * g + 3] = bv[3];
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const bf16x8 kf = *reinterpret_cast<const bf16x8*>(&ks_lds[sl][l32 * KROW + 16 * ks + 8 * hi]);
      sv = mfma32x32x16_t<F16>(kf, qf[ks], sv);
    }
    // Online softmax: running max, rescale, P in the operand format.
    float mx = sv[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, sv[r]);
    const float m_new = fmaxf(m, max_halves(mx) * c);
    const float alpha = __builtin_amdgcn_exp2f(m - m_new);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int db = 0; db < DB; ++db) o_acc[db] *= alpha;
    bf16x8 pb[2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[8 * s + e], c, -m));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[8 * s + e + 1], c, -m));
        l += p0 + p1;
        const bf16x2 pv2 = pack2<F16>(p0, p1);
        pb[s][e] = pv2[0];
        pb[s][e + 1] = pv2[1];
      }
    // O^T += V^T . P^T
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const bf16x8 vf =
            *reinterpret_cast<const bf16x8*>(&vt_lds[sl][(db * 32 + l32) * VROW + 16 * s + 8 * hi]);
        o_acc[db] = mfma32x32x16_t<F16>(vf, pb[s], o_acc[db]);
      }
    if (t + 1 < ntiles) store_tile(sl ^ 1);
  }

  const float l_tot = sum_halves(l);
  if (q_row >= p.M) return;
  const float inv = 1.0f / l_tot;
  uint16_t* O = p.o + b * p.o_sb + h * p.o_sh + q_row * p.o_sm;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int f0 = db * 32 + 8 * g + 4 * hi;             // features f0 .. f0+3
      if (f0 < HD) {
        const bf16x2 lo = pack2<F16>(o_acc[db][4 * g + 0] * inv, o_acc[db][4 * g + 1] * inv);
        const bf16x2 up = pack2<F16>(o_acc[db][4 * g + 2] * inv, o_acc[db][4 * g + 3] * inv);
        *reinterpret_cast<u32x2*>(O + f0) =
            u32x2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, up)};
      }
    }
  if (p.lse && hi == 0) p.lse[b * p.lse_sb + h * p.lse_sh + q_row] = m + __log2f(l_tot);
}

// ---------------------------------------------------------------------------
// Head dims 16 and 32, more than that: the narrow kernel.
//
// The VALU bounds it, not the matrix pipe: per wave and tile (64 queries x 32
// keys) 32 exps, 32 FMAs, 32 row-sum adds, 16 packs and 16 max3 are ~870
// cycles beside 256 (32) or 192 (16) MFMA cycles.  So everything else is kept
// off it:
//   * Two 32-query blocks per wave (256 queries per workgroup, three waves
//     per SIMD): every K and V fragment, bias read, DMA, wait and barrier
//     serves both.
//   * The offset is the exact running row max, as in the reference: a row's
//     largest P is exactly 1 and carries no rounding, which an offset fixed
//     from the first tiles gives up (error against 64 bits 2.35e-3 instead of
//     2.26e-3 in bf16, for 272 instead of 328 us at the sizes below).  Each
//     lane keeps the max of its own 16 keys; only where some row of a block
//     rose do the two lane halves meet and O and the row sums get rescaled,
//     in a wave-uniform branch per block (one branch for both: 331 us).
// K rows are XOR-swizzled in 16-byte chunks so that 16 consecutive keys hit 16
// distinct bank groups; a transposing V read covers 256 (128) consecutive
// bytes.  16 heads, 16,488 queries, 4,993 keys, against a kernel of one block
// per wave that transposed V with 2-byte LDS stores: 32 bf16 378 -> 328 us
// (82,440 queries, 23,939 keys: 6.72 -> 5.22 ms; 2,748 x 1,703: 48 -> 39 us),
// 16 bf16 342 -> 302 us, 32 fp16 388 -> 337 us.
constexpr int kNQ = kAWaves * 64;             // queries per workgroup

template <int HD>
struct NarrowSlot {
  uint16_t k[kAKT * HD];
  uint16_t v[kAKT * HD];
  float b[64];
};

template <int HD>
__device__ __forceinline__ int narrow_k_chunk(int key, int ch) {
  return HD == 32 ? ch ^ ((key >> 2) & 3) : ch ^ ((key >> 3) & 1);
}

// Workgroup barrier that leaves the DMAs of later tiles in flight; lgkmcnt(0)
// retires this wave's LDS reads before any slot is refilled.
__device__ __forceinline__ void ring_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int HD, bool F16>
__global__ __launch_bounds__(kAThreads, 3) void attn_narrow_kernel(AnyDimArgs p) {
  constexpr int KS = HD / 16;                 // k-steps of the score product
  constexpr int CH = HD / 8;                  // 16-byte chunks per key row
  constexpr int TW = kAKT * CH / 64;          // 16-byte DMAs (64 lanes) per tile and tensor
  constexpr int OPS = 2;                      // DMA instructions per wave and tile
  static_assert(HD < 64 && 2 * TW <= kAWaves, "one K or V DMA per wave and tile");
  __shared__ __attribute__((aligned(16))) NarrowSlot<HD> r0, r1, r2, r3;
  __shared__ __attribute__((aligned(16))) float b_sink[64];
  __shared__ __attribute__((aligned(16))) uint16_t kv_sink[2 * TW < kAWaves ? 512 : 8];

  const int tid = threadIdx.x, lane = tid & 63, hi = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int qb, bhi;
  {
    const uint32_t T = gridDim.x * gridDim.y, L = blockIdx.y * gridDim.x + blockIdx.x;
    const uint32_t q8 = T / 8, r8 = T % 8, x = L % 8;
    const uint32_t item = x * q8 + (x < r8 ? x : r8) + L / 8;
    qb = (int)(item % gridDim.x);
    bhi = (int)(item / gridDim.x);
  }
  const int64_t bh = bhi, b = bh / p.H, h = bh % p.H;
  const int64_t q_row = (int64_t)qb * kNQ + wave * 64 + l32;   // of block 0; block 1: + 32
  const uint16_t* Q = p.q + b * p.q_sb + h * p.q_sh;
  const uint16_t* K = p.k + b * p.k_sb + h * p.k_sh;
  const uint16_t* V = p.v + b * p.v_sb + h * p.v_sh;
  const int ntiles = (int)((p.N + kAKT - 1) / kAKT);
  const float* Brow = p.ws + bh * (int64_t)ntiles * kAKT;
  const float c = p.c;

  bf16x8 qf[2][KS];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[j][ks] = q_row + 32 * j < p.M ? *reinterpret_cast<const bf16x8*>(
                                             Q + (q_row + 32 * j) * p.q_sm + 16 * ks + 8 * hi)
                                       : bf16x8{};
  __builtin_amdgcn_sched_barrier(0);

  // The first TW waves fetch the tile's K, the next TW its V; at head dim 16
  // waves 2 and 3 point past the range into a sink, so that every wave issues
  // and waits for the same instructions.
  const bool is_k = wave < TW, sink = wave >= 2 * TW;
  const uint32_t kv_row = sink ? 0u : (uint32_t)(is_k ? p.k_sn : p.v_sn) * 2u;
  const __amdgpu_buffer_rsrc_t kvrs =
      make_rsrc(is_k ? K : V, (uint32_t)((p.N - 1) * (is_k ? p.k_sn : p.v_sn) * 2 + HD * 2));
  const __amdgpu_buffer_rsrc_t brs = make_rsrc(Brow, (uint32_t)ntiles * kAKT * 4u);
  const int part = wave % TW;                 // this wave's 64 chunks of the tensor's tile
  const int d_key = (part * 64 + lane) / CH, d_pch = (part * 64 + lane) % CH;
  const int d_ch = is_k ? narrow_k_chunk<HD>(d_key, d_pch) : d_pch;
  const uint32_t kv_voff = sink ? 0x80000000u : d_key * kv_row + (uint32_t)(d_ch * 16);
  const uint32_t b_voff = (wave == 0 && lane < kAKT) ? (uint32_t)lane * 4u : 0x40000000u;
  auto issue = [&](int t, NarrowSlot<HD>& S) {
    const uint32_t n0 = (uint32_t)t * kAKT;
    uint16_t* to = is_k ? &S.k[part * 512] : &S.v[part * 512];
    if (2 * TW < kAWaves && sink) to = &kv_sink[0];
    lds_dma16(kvrs, to, kv_voff, n0 * kv_row);
    float* dst = wave == 0 ? &S.b[0] : &b_sink[0];
    lds_dma4(brs, dst, b_voff, n0 * 4u);
  };

  int k_off[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) k_off[ks] = l32 * HD + (narrow_k_chunk<HD>(l32, 2 * ks + hi) << 3);
  // V^T operand as in attn_tiled_kernel.  (At head dim 16 the upper 16
  // features of the block repeat the lower ones and are never stored.)
  const int v_off = (4 * hi + ((lane & 15) >> 2)) * HD +
                    (2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) % CH * 8 + (lane & 1) * 4;

  auto scores = [&](const NarrowSlot<HD>& S, f32x16 (&sv)[2]) {
    f32x16 bias16;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 bv = *reinterpret_cast<const f32x4*>(&S.b[8 * g + 4 * hi]);
      bias16[4 * g + 0] = bv[0];
      bias16[4 * g + 1] = bv[1];
      bias16[4 * g + 2] = bv[2];
      bias16[4 * g + 3] = bv[3];
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const bf16x8 kf = *reinterpret_cast<const bf16x8*>(&S.k[k_off[ks]]);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        sv[j] = mfma32x32x16_t<F16>(kf, qf[j][ks], ks == 0 ? bias16 : sv[j]);
    }
  };
  // This lane's largest score of a block (its 16 of the row's 32 keys).
  auto lane_max = [&](const f32x16& x) {
    float mx = fmaxf(fmaxf(x[0], x[1]), x[2]);
#pragma unroll
    for (int r = 3; r < 15; r += 2) mx = fmaxf(fmaxf(mx, x[r]), x[r + 1]);
    return fmaxf(mx, x[15]);
  };

  f32x16 o_acc[2];
  f32x4 l[2];                                 // row sums in four parts
  float m[2], mx[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    l[j] = f32x4{};
    o_acc[j] = f32x16{};
  }

  issue(0, r0);
  issue(1, r1);
  issue(2, r2);
  wait_vmem<2 * OPS>();
  ring_barrier();
  f32x16 s_cur[2], s_nxt[2];
  scores(r0, s_cur);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    mx[j] = lane_max(s_cur[j]);
    m[j] = fmaxf(max_halves(mx[j]) * c, -1.0e30f);   // finite: a tile of -inf biases scores 0
  }

  // Iteration t: tile t in `cur`, tile t+1 in `nxt`, tile t+3 issued into
  // `dst` (the slot of tile t-1, free once every wave passed the barrier).
  auto iter = [&](int t, const NarrowSlot<HD>& cur, const NarrowSlot<HD>& nxt, NarrowSlot<HD>& dst) {
    wait_vmem<OPS>();                         // tile t+1 landed (tile t+2 in flight)
    ring_barrier();                           // ... for every wave
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (__builtin_amdgcn_ballot_w64(mx[j] * c > m[j]) != 0) {
        const float top = max_halves(mx[j]) * c;
        const float m_new = top > m[j] ? top : m[j];
        const float alpha = __builtin_amdgcn_exp2f(m[j] - m_new);
        m[j] = m_new;
        l[j] *= alpha;
        o_acc[j] *= alpha;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    issue(t + 3, dst);
    scores(nxt, s_nxt);
    bf16x8 vf[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      typedef short i16x4 __attribute__((ext_vector_type(4)));
      const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) i16x4*)&cur.v[v_off + 16 * s * HD]);
      const i16x4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) i16x4*)&cur.v[v_off + (16 * s + 8) * HD]);
      const bf16x4 l4 = __builtin_bit_cast(bf16x4, lo), u4 = __builtin_bit_cast(bf16x4, up);
      vf[s] = bf16x8{l4[0], l4[1], l4[2], l4[3], u4[0], u4[1], u4[2], u4[3]};
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      bf16x8 pb[2];
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s_cur[j][8 * s + e], c, -m[j]));
          const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s_cur[j][8 * s + e + 1], c, -m[j]));
          l[j][e & 2] += p0;
          l[j][(e & 2) + 1] += p1;
          const bf16x2 pv2 = pack2<F16>(p0, p1);
          pb[s][e] = pv2[0];
          pb[s][e + 1] = pv2[1];
        }
      // O^T += V^T . P^T
#pragma unroll
      for (int s = 0; s < 2; ++s) o_acc[j] = mfma32x32x16_t<F16>(vf[s], pb[s], o_acc[j]);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      mx[j] = lane_max(s_nxt[j]);
      s_cur[j] = s_nxt[j];
    }
    // (Operands of an empty asm: they stay in this iteration, and the
    // accumulators in place; without it the allocator copies them and spills.)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      asm volatile("" : "+v"(s_cur[j]), "+v"(l[j]), "+v"(o_acc[j]));
    __builtin_amdgcn_sched_barrier(0);
  };
  int t = 0;
  for (; t + 4 <= ntiles; t += 4) {
    iter(t, r0, r1, r3);
    iter(t + 1, r1, r2, r0);
    iter(t + 2, r2, r3, r1);
    iter(t + 3, r3, r0, r2);
  }
  if (t < ntiles) iter(t, r0, r1, r3);
  if (t + 1 < ntiles) iter(t + 1, r1, r2, r0);
  if (t + 2 < ntiles) iter(t + 2, r2, r3, r1);
  wait_vmem<0>();                             // no DMA may land after the workgroup ends

#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int64_t row = q_row + 32 * j;
    const float l_tot = sum_halves((l[j][0] + l[j][1]) + (l[j][2] + l[j][3]));
    if (row >= p.M) continue;
    const float inv = 1.0f / l_tot;
    uint16_t* O = p.o + b * p.o_sb + h * p.o_sh + row * p.o_sm;
#pragma unroll
    for (int g = 0; g < CH; ++g) {                           // features 8g + 4hi .. +3
      const bf16x2 lo = pack2<F16>(o_acc[j][4 * g + 0] * inv, o_acc[j][4 * g + 1] * inv);
      const bf16x2 up = pack2<F16>(o_acc[j][4 * g + 2] * inv, o_acc[j][4 * g + 3] * inv);
      *reinterpret_cast<u32x2*>(O + 8 * g + 4 * hi) =
          u32x2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, up)};
    }
    if (p.lse && hi == 0) p.lse[b * p.lse_sb + h * p.lse_sh + row] = m[j] + __log2f(l_tot);
  }
}

// Whether the short kernel is the faster one at head dims 16 and 32.  Its line
// in keys falls as the chip fills up: past four of its workgroups per CU its
// slower tile counts from 192 keys on, past one from 512; below, a call is one
// workgroup's walk and the other kernel's pre-pass and wider waves pay off only
// from 2,048 keys (no bias and at most half the CUs busy: 4,096), or from 1,024
// where many heads' K and V compete for the L2s.  Measured over 4 to 128 heads,
// 1 to 8,000 queries and 32 to 20,000 keys in both formats: the kernel
// taken is never over 1.14 times the better one's time, 1.002 times on average.
bool short_call(const AnyDimArgs& a, int64_t D, int bias_kind) {
  const int64_t groups = (a.M + kAQ - 1) / kAQ * a.BH;
  if (groups > 1024) return a.N <= 192;
  if (groups > 256) return a.N <= 512;
  if (a.BH * D > 2048) return a.N <= 1024;
  return a.N <= (bias_kind == GPA_BIAS_NONE && groups <= 128 ? 4096 : 2048);
}

template <int HD, bool F16>
void launch_short(const AnyDimArgs& a, int bias_kind, hipStream_t s) {
  const dim3 grid((unsigned)((a.M + kAQ - 1) / kAQ), (unsigned)(a.BH)), block(kAThreads);
  switch (bias_kind) {
    case GPA_BIAS_F32:
      hipLaunchKernelGGL((attn_short_kernel<HD, F16, GPA_BIAS_F32>), grid, block, 0, s, a);
      break;
    case GPA_BIAS_BF16:
      hipLaunchKernelGGL((attn_short_kernel<HD, F16, GPA_BIAS_BF16>), grid, block, 0, s, a);
      break;
    case GPA_BIAS_F16:
      hipLaunchKernelGGL((attn_short_kernel<HD, F16, GPA_BIAS_F16>), grid, block, 0, s, a);
      break;
    default:
      hipLaunchKernelGGL((attn_short_kernel<HD, F16, GPA_BIAS_NONE>), grid, block, 0, s, a);
      break;
  }
}

template <int HD, bool F16>
hipError_t launch_hd(const AnyDimArgs& a, int bias_kind, hipStream_t s) {
  if constexpr (HD < 64) {
    if (short_call(a, HD, bias_kind)) {
      launch_short<HD, F16>(a, bias_kind, s);
      return hipGetLastError();
    }
  }
  const int64_t ntiles = (a.N + kAKT - 1) / kAKT, npad = ntiles * kAKT;
  const dim3 bgrid((unsigned)((npad + 255) / 256), (unsigned)a.BH), bblock(256);
  switch (bias_kind) {
    case GPA_BIAS_F32:
      hipLaunchKernelGGL((bias_rows_kernel<GPA_BIAS_F32>), bgrid, bblock, 0, s, a.bias, a.ws, a.H,
                         a.N, npad, a.bias_sb, a.bias_sh, a.bias_sn, a.mul);
      break;
    case GPA_BIAS_BF16:
      hipLaunchKernelGGL((bias_rows_kernel<GPA_BIAS_BF16>), bgrid, bblock, 0, s, a.bias, a.ws, a.H,
                         a.N, npad, a.bias_sb, a.bias_sh, a.bias_sn, a.mul);
      break;
    case GPA_BIAS_F16:
      hipLaunchKernelGGL((bias_rows_kernel<GPA_BIAS_F16>), bgrid, bblock, 0, s, a.bias, a.ws, a.H,
                         a.N, npad, a.bias_sb, a.bias_sh, a.bias_sn, a.mul);
      break;
    default:
      hipLaunchKernelGGL((bias_rows_kernel<GPA_BIAS_NONE>), bgrid, bblock, 0, s, a.bias, a.ws,
                         a.H, a.N, npad, a.bias_sb, a.bias_sh, a.bias_sn, a.mul);
      break;
  }
  if constexpr (HD < 64) {
    const dim3 grid((unsigned)((a.M + kNQ - 1) / kNQ), (unsigned)(a.BH)), block(kAThreads);
    hipLaunchKernelGGL((attn_narrow_kernel<HD, F16>), grid, block, 0, s, a);
  } else {
    const dim3 grid((unsigned)((a.M + kAQ - 1) / kAQ), (unsigned)(a.BH)), block(kAThreads);
    hipLaunchKernelGGL((attn_tiled_kernel<HD, F16>), grid, block, 0, s, a);
  }
  return hipGetLastError();
}

}  // namespace

bool attn_any_dim_supported(int64_t D) { return D == 16 || D == 32 || D == 128 || D == 256; }

size_t attn_any_dim_ws_bytes(int64_t BH, int64_t N) {
    return (size_t)(BH * ((N + kAKT - 1) / kAKT) * kAKT) * sizeof(float);
}

template <bool F16>
hipError_t attn_any_dim_launch(const AnyDimArgs& a, int64_t D, int bias_kind, hipStream_t s) {
  switch (D) {
    case 16: return launch_hd<16, F16>(a, bias_kind, s);
    case 32: return launch_hd<32, F16>(a, bias_kind, s);
    case 128: return launch_hd<128, F16>(a, bias_kind, s);
    case 256: return launch_hd<256, F16>(a, bias_kind, s);
    default: return hipErrorInvalidValue;
  }
}

template hipError_t attn_any_dim_launch<false>(const AnyDimArgs&, int64_t, int, hipStream_t);
template hipError_t attn_any_dim_launch<true>(const AnyDimArgs&, int64_t, int, hipStream_t);

}  // namespace gpa
