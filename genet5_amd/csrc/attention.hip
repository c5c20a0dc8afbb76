// Varlen bidirectional attention with ALiBi on bf16 MFMA (gfx950).
//
// Reference interface: flash_attn_varlen_func(q, k, v, cu_seqlens_q,
// cu_seqlens_k, max_seqlen_q, max_seqlen_k, dropout_p, softmax_scale,
// causal=False) as GeneT5's FlashAttention.forward calls it
// (lib/blocks/_flash_att.py:60-98), with flash-attn's `alibi_slopes` bias
// bias[h, i, j] = -slope_h * |i - j| (sequence-local positions, non-causal,
// equal query and key lengths).  Sequences of the packed batch attend only
// within themselves (cu_seqlens), unlike the reference SDPA fallback's single
// global mask (lib/blocks/_sdpa_att.py:36-43).
//
// Work split: one workgroup of 4 waves per (128-query block, head, sequence);
// wave w owns queries q0 + 32w .. q0 + 32w + 31.  Keys stream through LDS in
// blocks of 64, a ring of three (K, V) tiles filled by LDS DMA (no staging
// registers, no LDS writes), one barrier per block: after the softmax, when the
// next tile has landed and every wave holds its V operands of this one; the next
// block's K operands are read behind the output product.  Each wave walks its
// blocks as runs of one kind (before its queries, across them, after them, the
// partial last one), so that the block loops carry no branches.
//
// What bounds it: issue and power.  With two waves per SIMD the matrix core and the
// VALU are each busy half of the cycles with ALiBi (counters, 8 x 4,550 tokens, 12
// heads: 50 and 51 %, at 1.98 GHz) and 60 and 57 % without (1.84 GHz under the power
// limit), no LDS bank conflicts; per 64-key block and wave 22 MFMAs (704 cycles)
// against 32 exps (8 cycles each), 32 multiplies, 16 conversions and about 30 more.
// Against the register-staged loop with a branch per block before it (and a
// multiplied-out bias in its online loop), the same calls on one GPU: 8 x 4,550
// tokens with ALiBi 402 -> 339 us, with twice the scores (online loop) 522 -> 456, no
// ALiBi 745 -> 592 (859 TFLOP/s); 2 x 3,000 without ALiBi 115 -> 86, 4 x 2,048 86 -> 74.
//
// MFMA layout (v_mfma_f32_32x32x16_bf16): scores are formed transposed,
// S^T = K . Q^T, with the key block as the A operand and the wave's queries as
// the B operand, so lane l holds query l % 32 and, in element 4q + u of key
// block b, key 32b + 8q + 4(l / 32) + u.  Every softmax statistic of a query
// lives in the two lanes l and l ^ 32; one cross-lane exchange per key block
// shares the block maximum and the row sums are combined once at the end.
// The output is formed transposed too, O^T += V^T . P^T: P^T needs no data
// movement (a lane's eight probabilities of a 16-key chunk are its own
// accumulator elements), provided V^T's key order inside each 16-key chunk is
// the one those elements carry: key r at position r with bits 2 and 3
// swapped.  V's transposing LDS reads fetch the keys in that order.
//
// LDS rows are 128 bytes, their 16-byte chunks swizzled by the row (see the tile
// loads) so that the fragment reads hit distinct banks.
//
// Block skipping under ALiBi: with key norms bounded by KM (the largest of the
// per-64-token-block maxima a pre-pass writes, over the blocks that cover the
// sequence) and the query norms of the workgroup by NQ,
// every score obeys |s| <= NQ * KM (Cauchy-Schwarz), so a key at distance
// > W = (2 * scale * log2(e) * NQ * KM + 64) / (slope * log2(e)) from every
// query of the workgroup has p < 2^-64 relative to the row's largest term
// (the diagonal key is always computed and bounds the row maximum from
// below).  The workgroup therefore visits only the key blocks within W of its
// queries; the skipped probability mass is below 2^-51 of each row's sum, so
// the result equals the dense computation to fp32 rounding.
//
// Softmax in base 2: t = s * scale * log2(e) + bias * log2(e).  Two loops:
//
// * Reference maximum (with key norms, a positive scale, a non-negative slope
//   and every |s * sc| of the workgroup within 32): p = 2^(t - mref) with the
//   lane's fixed upper bound mref = sc * |q| * KM >= t.  The row's largest term
//   is at least its diagonal's, >= -mref, so no probability that matters
//   underflows and no running maximum or rescaling is needed; the row sums that
//   normalise the output come from an all-ones MFMA operand against P^T
//   (the sums of the bf16 probabilities the output product weights; the fp32
//   sums are kept only when softmax_lse is asked for).
// * Online (otherwise): running maximum, rescaled output and row sum.
//
// On a key block wholly on one side of the wave's queries (and inside the
// sequence) the ALiBi bias (and the reference loop's -mref) enters the score
// product as one more MFMA k-chunk (key offsets against bf16 splits of the slope
// and of the lane's constant), so a probability costs one multiply (or fused
// multiply-add) and one exp.
//
// Blocks that straddle the diagonal or the sequence end take the exact
// per-element |i - j| path with masking in both loops.
#include <algorithm>
#include <type_traits>

#include "gemm_common.h"

namespace g5moe {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kHeadDim = 64;
constexpr int kBQ = 128;   // queries per workgroup (32 per wave)
constexpr int kBKV = 64;   // keys per LDS block
constexpr int kRowBytes = kHeadDim * 2;           // one key's K or V row in LDS
constexpr int kTileBytes = kBKV * kRowBytes;      // 8 KB
constexpr int kStageBytes = 2 * kTileBytes;       // K tile, then V tile
constexpr int kStages = 3;
constexpr float kSkipMargin = 64.0f;              // skipped keys have p < 2^-64
constexpr float kFixedGap = 64.0f;                // reference-max loop: row maximum >= 2^-64
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

struct AttnArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  const int32_t* cu_seqlens;  // [n_seqs + 1]
  int64_t q_tok, k_tok, v_tok, o_tok;      // element strides between tokens
  int64_t q_head, k_head, v_head, o_head;  // element strides between heads
  int group;                  // query heads per key/value head
  float sc;                   // softmax_scale * log2(e)
  const float* slopes;        // [n_heads] or nullptr
  float* lse;                 // [n_heads, total] (natural log) or nullptr
  const float* kmax;          // [n_kv_heads, ceil(total / 64)] largest key norm of each
                              // 64-token block, or nullptr (dense)
  int n_kblk;                 // ceil(total / 64)
  int64_t total;
};

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4* lds_i16x4_p;

// ds_read_b64_tr_b16 (gfx950): within each 16-lane group the lanes' 64-bit
// chunks form a 16 x 4 matrix (lane k's chunk is row k), and lane i receives
// element i % 4 of rows i / 4, 4 + i / 4, 8 + i / 4 and 12 + i / 4.
__device__ __forceinline__ i16x4 read_tr(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_i16x4_p>(
      uintptr_t((__attribute__((address_space(3))) const char*)p)));
}

// LDS DMA with a 64-bit address per lane (gemm::lds_dma16_s with a scalar base
// otherwise).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_dma16_v(const char* addr, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :: "v"(addr), "s"(__builtin_amdgcn_readfirstlane(lds))
               : "memory", "m0");
}
#pragma clang diagnostic pop

// LSE: softmax_lse is written (a.lse != nullptr).  WIDE: a token stride of k or v
// too large for 32-bit offsets inside a 64-key tile.  NEG: a negative scale, taken as
// its magnitude on negated queries (exactly the same products).
template <bool LSE, bool WIDE, bool NEG>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(2, 2)))
void attn_fwd_kernel(AttnArgs a) {
  __shared__ __attribute__((aligned(1024))) char ring[kStages * kStageBytes];

  const int z = blockIdx.z;
  const int hq = blockIdx.y;
  // Sequence bounds clamped to [0, total]: a malformed cu_seqlens cannot move
  // an access outside the q/k/v/out buffers.
  const int total = int(a.total);
  const int s0 = min(max(a.cu_seqlens[z], 0), total);
  const int L = min(max(a.cu_seqlens[z + 1], s0), total) - s0;
  const int q0 = blockIdx.x * kBQ;
  if (q0 >= L) return;
  const int hk = hq / a.group;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5;
  const int col = lane & 31;
  const int iq = q0 + wave * 32 + col;       // this lane's query (sequence position)
  const int wq_lo = q0 + wave * 32;          // the wave's query range
  const int wq_hi = wq_lo + 31;
  const float sl = a.slopes != nullptr ? a.slopes[hq] * kLog2e : 0.0f;
  const float sc = NEG ? -a.sc : a.sc;

  // Q^T operand: lane holds query iq, head dims 16kc + 8*half .. +8.
  bf16x8 qf[4];
  {
    const bool ok = iq < L;
    const uint16_t* qp = a.q + int64_t(s0 + (ok ? iq : 0)) * a.q_tok + hq * a.q_head + half * 8;
#pragma unroll
    for (int kc = 0; kc < 4; ++kc) {
      const u32x4 raw = ok ? *reinterpret_cast<const u32x4*>(qp + 16 * kc) : u32x4{0, 0, 0, 0};
      qf[kc] = __builtin_bit_cast(bf16x8, raw);
    }
    // the queries landed: a load the compiler still counted as in flight at the
    // block loop would make every block wait for its tile loads (vmcnt 0)
#pragma unroll
    for (int kc = 0; kc < 4; ++kc) {
      u32x4 w = __builtin_bit_cast(u32x4, qf[kc]);
      if constexpr (NEG) {
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] ^= 0x80008000u;
      }
      asm volatile("" : "+v"(w));
      qf[kc] = __builtin_bit_cast(bf16x8, w);
    }
  }
  // Key blocks this workgroup visits: [n_lo, n_hi] (all of them without ALiBi
  // or without key norms).  With key norms, `fixed` selects the reference-max
  // loop when every score term s * sc of the workgroup is provably within
  // kFixedGap / 2 of zero; mref is then this lane's upper bound on its row's
  // largest term.
  const int nblk = (L + kBKV - 1) / kBKV;
  int n_lo = 0, n_hi = nblk - 1;
  bool fixed = false;
  float mref = 0.0f;
  if (a.kmax != nullptr) {
    __shared__ float red[8];
    // largest key norm over the 64-token blocks that cover the sequence
    float km = 0.0f;
    const float* bm = a.kmax + int64_t(hk) * a.n_kblk;
    for (int i = (s0 >> 6) + tid; i <= ((s0 + L - 1) >> 6); i += 256) km = __builtin_fmaxf(km, bm[i]);
#pragma unroll
    for (int bit = 32; bit >= 1; bit >>= 1) km = __builtin_fmaxf(km, __shfl_xor(km, bit, 64));
    float ss = 0.0f;
#pragma unroll
    for (int kc = 0; kc < 4; ++kc)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = float(qf[kc][e]);
        ss = __builtin_fmaf(x, x, ss);
      }
    ss += __shfl_xor(ss, 32, 64);
    const float ss_own = ss;  // this lane's squared query norm
#pragma unroll
    for (int bit = 16; bit >= 1; bit >>= 1) ss = __builtin_fmaxf(ss, __shfl_xor(ss, bit, 64));
    if (lane == 0) {
      red[wave] = ss;
      red[4 + wave] = km;
    }
    __syncthreads();
    const float nq2 = __builtin_fmaxf(__builtin_fmaxf(red[0], red[1]), __builtin_fmaxf(red[2], red[3]));
    const float kmx = __builtin_fmaxf(__builtin_fmaxf(red[4], red[5]), __builtin_fmaxf(red[6], red[7]));
    // |s * sc| <= bound for every query of the workgroup and key of the sequence
    const float bound = __builtin_fabsf(sc) * __builtin_sqrtf(nq2) * kmx;
    if (sl > 0.0f) {
      const float w = (2.0f * bound + kSkipMargin) / sl;
      if (w < 1.0e9f) {  // false for inf / NaN: visit every block
        const int wi = int(w);
        const int q_hi = min(q0 + kBQ, L) - 1;
        n_lo = max(0, (q0 - wi) / kBKV);
        n_hi = min(nblk - 1, (q_hi + wi) / kBKV);
      }
    }
    // bound is the same in every lane (red); false for inf / NaN.  sl < 2^60 sc
    // keeps the slope in units of raw scores (u = sl / sc) and its products
    // with key offsets and distances (< 2^31) finite.
    fixed = __builtin_amdgcn_readfirstlane(int(!NEG && sc > 0.0f && sl >= 0.0f && sl < sc * 0x1p60f &&
                                               2.0f * bound <= kFixedGap)) != 0;
    mref = sc * __builtin_sqrtf(ss_own) * kmx;
  }

  // Tile loads, straight to LDS: DMA instruction i (0, 1: K, 2, 3: V) of a wave
  // fills the 8 key rows of block 4 (i % 2) + wave of a tile.  K's chunk c of row r
  // goes to c ^ ((r >> 1) & 7) (16-lane groups of a fragment read then hit 16
  // distinct bank groups), V's to c ^ 2 (r & 3) (the four keys of a transposing
  // read in four distinct ones).  Rows past the sequence end repeat its last row:
  // their scores are masked, and V's are cleared before they are read.
  const int lrow = lane >> 3;
  const uint32_t k_ch = uint32_t((lane & 7) ^ (((wave & 1) * 4 + (lrow >> 1)) & 7)) * 16;
  const uint32_t v_ch = uint32_t((lane & 7) ^ (2 * (lrow & 3))) * 16;
  const char* const kbase =
      reinterpret_cast<const char*>(a.k + int64_t(s0) * a.k_tok + hk * a.k_head);
  const char* const vbase =
      reinterpret_cast<const char*>(a.v + int64_t(s0) * a.v_tok + hk * a.v_head);
  const int64_t k_tok2 = a.k_tok * 2, v_tok2 = a.v_tok * 2;
  const uint32_t ring_lds = gemm::lds_addr(ring) + uint32_t(wave) * 1024;
  // Lane offsets of the wave's rows in a whole tile and in the sequence's last one.
  const int last_rows = L - (nblk - 1) * kBKV;
  uint32_t koff[2][2], voff[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = (4 * i + wave) * 8 + lrow;
    koff[0][i] = uint32_t(row) * uint32_t(k_tok2) + k_ch;
    voff[0][i] = uint32_t(row) * uint32_t(v_tok2) + v_ch;
    const int rl = min(row, last_rows - 1);
    koff[1][i] = uint32_t(rl) * uint32_t(k_tok2) + k_ch;
    voff[1][i] = uint32_t(rl) * uint32_t(v_tok2) + v_ch;
  }
  // The next tile to load (n_is, at kt / vt); past n_hi the last tile goes out
  // again, into a buffer that no later block reads, so that every block issues
  // four instructions and the waits are constants.
  int n_is = n_lo;
  const char* kt = kbase + n_lo * kBKV * k_tok2;
  const char* vt = vbase + n_lo * kBKV * v_tok2;
  auto issue = [&](uint32_t boff) __attribute__((always_inline)) {
    const uint32_t dst = ring_lds + boff;
    const bool last = n_is == nblk - 1;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if constexpr (WIDE) {
        const int r0 = (4 * i + wave) * 8 + lrow;
        const int row = last ? min(r0, last_rows - 1) : r0;
        lds_dma16_v(kt + row * k_tok2 + k_ch, dst + i * 4096);
        lds_dma16_v(vt + row * v_tok2 + v_ch, dst + kTileBytes + i * 4096);
      } else {
        gemm::lds_dma16_s(kt, last ? koff[1][i] : koff[0][i], dst + i * 4096);
        gemm::lds_dma16_s(vt, last ? voff[1][i] : voff[0][i], dst + kTileBytes + i * 4096);
      }
    }
    const bool more = n_is < n_hi;
    n_is += more ? 1 : 0;
    kt += more ? kBKV * k_tok2 : 0;
    vt += more ? kBKV * v_tok2 : 0;
  };
  // K fragments of a block: keys 32 b + col, head dims 16 kc + 8 half .. + 8
  const int k_row = col * kRowBytes;
  const int k_sw = (col >> 1) & 7;
  bf16x8 kf[2][4];
  auto load_kf = [&](uint32_t boff) __attribute__((always_inline)) {
    const char* Ks = ring + boff + k_row;
#pragma unroll
    for (int kc = 0; kc < 4; ++kc)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        kf[b][kc] = *reinterpret_cast<const bf16x8*>(Ks + 32 * b * kRowBytes +
                                                     ((2 * kc + half) ^ k_sw) * 16);
  };
  // S^T = K . Q^T for the two 32-key halves of the block
  auto scores = [&](f32x16* s) __attribute__((always_inline)) {
    const f32x16 zero16 = {};
#pragma unroll
    for (int kc = 0; kc < 4; ++kc)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        s[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[b][kc], qf[kc], kc == 0 ? zero16 : s[b],
                                                       0, 0, 0);
  };
  // P^T operand of 16-key chunk c (chunk c = key block c / 2, elements
  // 8 (c % 2) .. +8): the lane's own probabilities, no data movement
  auto p_chunk = [&](const uint32_t (*pk)[8], int c) __attribute__((always_inline)) -> bf16x8 {
    const u32x4 praw = {pk[c >> 1][4 * (c & 1) + 0], pk[c >> 1][4 * (c & 1) + 1],
                        pk[c >> 1][4 * (c & 1) + 2], pk[c >> 1][4 * (c & 1) + 3]};
    return __builtin_bit_cast(bf16x8, praw);
  };
  // The V^T operand of lane (col, half) for chunk c is head dim 32 mb + col at the
  // keys its P^T elements hold, 16 c + 4 half + {0..3, 8..11}: two transposing
  // reads of four keys each, lane k of a 16-lane group addressing key (k / 4) of
  // the four and the four dims from 4 (k % 4) of the group's 16, i.e. byte
  // 8 (k % 2) of chunk 4 mb + 2 (group % 2) + (k % 4) / 2.  The chunk's swizzle
  // 2 (key % 4) = 2 (k / 4) is the lane's own.
  const int vk = (lane & 15) >> 2;
  const int v_row = kTileBytes + (4 * half + vk) * kRowBytes + 8 * (lane & 1);
  const int v_c = (2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ (2 * vk);
  const int v_lane[2] = {v_row + v_c * 16, v_row + (v_c ^ 4) * 16};
  bf16x8 vf[4][2];
  auto load_vf = [&](uint32_t boff) __attribute__((always_inline)) {
    const char* Vs = ring + boff;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) {
        const char* vp = Vs + v_lane[mb] + 16 * c * kRowBytes;
        const i16x4 lo = read_tr(vp);
        const i16x4 hi = read_tr(vp + 8 * kRowBytes);
        const i16x4 vv[2] = {lo, hi};
        vf[c][mb] = __builtin_bit_cast(bf16x8, vv);
      }
  };
  // Exact per-element bias and sequence-end mask of a block that straddles the
  // wave's queries or the sequence end: t = s * sc - sl * |i - j|, -inf past L.
  auto exact_terms = [&](f32x16* s, int j0) __attribute__((always_inline)) {
    // distances and limits from the lane's first key, so that each element's own
    // offset is a literal
    const float di = float(iq - j0 - 4 * half);
    const int lim = L - j0 - 4 * half;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kr = 32 * b + 8 * (r >> 2) + (r & 3);
        const float bias = -sl * __builtin_fabsf(di - float(kr));
        s[b][r] = kr < lim ? __builtin_fmaf(s[b][r], sc, bias) : -__builtin_inff();
      }
  };

  f32x16 o[2] = {f32x16{}, f32x16{}};
  // reference maximum, normalising sum, fp32 sum for lse
  float m = fixed ? mref : -__builtin_inff(), l_tot = 0.0f, l_lse = 0.0f;

  // The ALiBi bias of a block wholly on one side of the wave's queries as one more
  // 16-deep MFMA chunk, in units of raw scores: key rows [kr, kr, kr, 1, 1, 1, 0, 0]
  // (kr the key's offset in the block, exact in bf16; the other half zero) against
  // query columns [-+u1, -+u2, -+u3, c1, c2, c3, 0, 0], where u1 + u2 + u3 = u =
  // sl / sc and c1 + c2 + c3 = c = -u |j0 - i| (the reference-max loop: - mref / sc)
  // are bf16 splits, exact to fp32 precision (bf16 products are exact in the fp32
  // accumulation).  Per block only c's words change.  Slopes and scales of either sign
  // take it; a scale of 0 or a slope out of range makes every block exact (8 x 4,550
  // tokens, 12 heads, this against every block exact: ALiBi's slopes times -0.01 679
  // against 790 us, a scale of -0.125 without a bias 656 against 792).
  const bool chunk_ok = __builtin_amdgcn_readfirstlane(
                            int(sc > 0.0f && __builtin_fabsf(sl) < sc * 0x1p60f)) != 0;
  auto bf16r = [](float x) __attribute__((always_inline)) -> float { return float(__bf16(x)); };
  const uint32_t half0 = half == 0 ? 0xffffffffu : 0u;
  const float u = chunk_ok ? sl / sc : 0.0f;
  const float mref_s = fixed ? mref / sc : 0.0f;
  u32x4 kx[2];      // key rows of the two 32-key halves
  uint32_t qu[3];   // [u1, u2], [u3, 0] and the sign bits of both (keys after: minus)
  {
    const float u1 = bf16r(u), u2 = bf16r(u - u1), u3 = bf16r(u - u1 - u2);
    qu[0] = pack_bf16x2(u1, u2) & half0;
    qu[1] = pack_bf16x2(u3, 0.0f) & half0;
    qu[2] = 0x80008000u & half0;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const float kr = float(32 * b + col);
      kx[b] = u32x4{pack_bf16x2(kr, kr) & half0, pack_bf16x2(kr, 1.0f) & half0,
                    pack_bf16x2(1.0f, 1.0f) & half0, 0u};
    }
  }
  // Adds the chunk; dist = |j0 - i|, qw: the signed u words of the block's side
  auto add_chunk = [&](f32x16* s, float dist, const uint32_t (&qw)[2])
      __attribute__((always_inline)) {
    const float c = -u * dist - mref_s;
    const float c1 = bf16r(c), c2 = bf16r(c - c1), c3 = bf16r(c - c1 - c2);
    // (the other half's key rows are zero: its query columns only have to be finite)
    const u32x4 q = {qw[0], qw[1] | (__float_as_uint(c1) & 0xffff0000u), pack_bf16x2(c2, c3), 0u};
#pragma unroll
    for (int b = 0; b < 2; ++b)
      s[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kx[b]),
                                                     __builtin_bit_cast(bf16x8, q), s[b], 0, 0, 0);
  };
  auto block_max = [](const f32x16* s) __attribute__((always_inline)) -> float {
    float mx = s[0][0];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; r += 2)
        mx = __builtin_fmaxf(__builtin_fmaxf(mx, s[b][r]), s[b][r + 1]);
    return mx;
  };

  // The wave's blocks [n_lo, n_hi] in order: [n_lo, e0) and [e1, e2) by the fast
  // path (whole blocks on one side of the wave's queries, or any whole block
  // without ALiBi), [e0, e1) and a partial last block by the exact one.  Every
  // wave of the workgroup runs every block, so the barriers pair up.
  const int end = min(n_hi + 1, L / kBKV);
  int e0, e1;
  if (!chunk_ok) {
    e0 = n_lo;
    e1 = end;
  } else if (sl == 0.0f) {
    e0 = e1 = end;
  } else {
    e0 = min(wq_lo / kBKV, end);
    e1 = min(wq_lo / kBKV + 1, end);
  }
  const bool tail = n_hi == nblk - 1 && last_rows < kBKV;

  uint32_t boff = 0;
#pragma unroll
  for (int st = 0; st < kStages; ++st) issue(uint32_t(st) * kStageBytes);
  gemm::wait_vmcnt<(kStages - 1) * 4>();
  __syncthreads();
  load_kf(0);

  auto run = [&](auto fixed_c, auto chunk_c) __attribute__((always_inline)) {
    constexpr bool FIXED = decltype(fixed_c)::value;
    constexpr bool CHUNK = decltype(chunk_c)::value;
    const __bf16 b1 = __bf16(1.0f);
    const bf16x8 ones = {b1, b1, b1, b1, b1, b1, b1, b1};
    f32x16 lacc = {};   // FIXED: sums of the bf16 probabilities, which normalise the output
    float psum = 0.0f;  // fp32 sums (FIXED: for lse only)
    // Online: the running maximum; a new one rescales the output and the sum
    auto advance = [&](float mx) __attribute__((always_inline)) {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx),
                                                       false, false);
      mx = __builtin_fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      const float m_new = __builtin_fmaxf(m, mx);
      if (__ballot(m_new != m) != 0) {
        const float alpha = __builtin_amdgcn_exp2f(m - m_new);
        m = m_new;
        psum *= alpha;
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[mb][r] *= alpha;
      }
    };
    // One block; EXACT: per-element bias and mask, n its number; else dist and qw as
    // add_chunk takes them.
    auto step = [&](auto exact_c, int n, float dist, const uint32_t (&qw)[2])
        __attribute__((always_inline)) {
      constexpr bool EXACT = decltype(exact_c)::value;
      f32x16 s[2];
      scores(s);
      load_vf(boff);
      if constexpr (EXACT) {
        exact_terms(s, n * kBKV);
        if constexpr (!FIXED) advance(block_max(s));
      } else {
        if constexpr (CHUNK) add_chunk(s, dist, qw);
        if constexpr (!FIXED) advance(block_max(s) * sc);
      }
      uint32_t pk[2][8];
      float sum = 0.0f;
      auto term = [&](int b, int r) __attribute__((always_inline)) -> float {
        if constexpr (EXACT)
          return s[b][r] - m;
        else if constexpr (FIXED && CHUNK)
          return s[b][r] * sc;  // the chunk carries -m
        else
          return __builtin_fmaf(s[b][r], sc, -m);
      };
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          const float p0 = __builtin_amdgcn_exp2f(term(b, r));
          const float p1 = __builtin_amdgcn_exp2f(term(b, r + 1));
          if constexpr (!FIXED || LSE) {
            sum += p0;
            sum += p1;
          }
          pk[b][r >> 1] = pack_bf16x2(p0, p1);
        }
      if constexpr (!FIXED || LSE) psum += sum;
      // the next stage landed, and every wave has read all of this one
      gemm::wait_vmcnt<(kStages - 2) * 4>();
      __syncthreads();
      issue(boff);
      boff = boff + kStageBytes == kStages * kStageBytes ? 0 : boff + kStageBytes;
      load_kf(boff);
      // O^T += V^T . P^T over the four 16-key chunks
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const bf16x8 pf = p_chunk(pk, c);
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
          o[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[c][mb], pf, o[mb], 0, 0, 0);
        if constexpr (FIXED)
          lacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, pf, lacc, 0, 0, 0);
      }
    };
    using T_ = std::true_type;
    using F_ = std::false_type;
    // the query's distance to the block's first key, exact in fp32
    const uint32_t q_before[2] = {qu[0], qu[1]};
    const uint32_t q_after[2] = {qu[0] ^ qu[2], qu[1] ^ (qu[2] & 0xffffu)};
    int n = n_lo;
    float dist = float(iq - n_lo * kBKV);
    for (; n < e0; ++n, dist -= float(kBKV)) step(F_{}, n, dist, q_before);
    for (; n < e1; ++n, dist -= float(kBKV)) step(T_{}, n, 0.0f, q_before);
    dist = -dist;
    for (; n < end; ++n, dist += float(kBKV)) step(F_{}, n, dist, q_after);
    if (tail) {
      // V rows past the sequence end: 0 (times a masked key's 0 probability)
      for (int i = tid; i < (kBKV - last_rows) * 8; i += 256)
        *reinterpret_cast<u32x4*>(ring + boff + kTileBytes + last_rows * kRowBytes + i * 16) =
            u32x4{0, 0, 0, 0};
      __syncthreads();
      step(T_{}, n, 0.0f, q_before);
    }
    l_lse = psum + __shfl_xor(psum, 32, 64);
    l_tot = FIXED ? lacc[0] : l_lse;
  };
  if (fixed && sl != 0.0f)
    run(std::true_type{}, std::true_type{});
  else if (fixed)
    run(std::true_type{}, std::false_type{});
  else if (sl != 0.0f)
    run(std::false_type{}, std::true_type{});
  else
    run(std::false_type{}, std::false_type{});
  // refills past the last block may still be landing in this workgroup's LDS
  gemm::wait_vmcnt<0>();

  // normalise and store: lane holds query iq, dims 32mb + 8q + 4half + u
  if (iq < L) {
    const float inv = 1.0f / l_tot;
    uint16_t* op = a.o + int64_t(s0 + iq) * a.o_tok + hq * a.o_head + 4 * half;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        uint2 w;
        w.x = pack_bf16x2(o[mb][4 * q] * inv, o[mb][4 * q + 1] * inv);
        w.y = pack_bf16x2(o[mb][4 * q + 2] * inv, o[mb][4 * q + 3] * inv);
        *reinterpret_cast<uint2*>(op + 32 * mb + 8 * q) = w;
      }
    if (LSE && half == 0)
      a.lse[int64_t(hq) * a.total + s0 + iq] = (m + __builtin_log2f(l_lse)) * kLn2;
  }
}

// Largest key norm of each 64-token block of each key/value head:
// kmax[h * n_kblk + b] = max over tokens t in [64b, 64b + 64) of ||k[t, h]||
// (fp32).  One workgroup per (block, head); eight lanes per 128-byte key row.
__global__ __launch_bounds__(256) void key_norm_max_kernel(const uint16_t* __restrict__ k,
                                                           int64_t k_tok, int64_t k_head,
                                                           int64_t total, int n_kblk,
                                                           float* kmax) {
  __shared__ float red[4];
  const int b = blockIdx.x, h = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int chunk = tid & 7;
  float best = 0.0f;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int64_t t = int64_t(b) * 64 + pass * 32 + (tid >> 3);
    float ss = 0.0f;
    if (t < total) {
      const u32x4 raw = *reinterpret_cast<const u32x4*>(k + t * k_tok + h * k_head + chunk * 8);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float lo = bf16_bits_to_f32(raw[w] & 0xffffu);
        const float hi = bf16_bits_to_f32(raw[w] >> 16);
        ss = __builtin_fmaf(lo, lo, ss);
        ss = __builtin_fmaf(hi, hi, ss);
      }
    }
    ss += __shfl_xor(ss, 1, 64);
    ss += __shfl_xor(ss, 2, 64);
    ss += __shfl_xor(ss, 4, 64);
    best = __builtin_fmaxf(best, ss);
  }
#pragma unroll
  for (int bit = 8; bit <= 32; bit <<= 1) best = __builtin_fmaxf(best, __shfl_xor(best, bit, 64));
  if (lane == 0) red[tid >> 6] = best;
  __syncthreads();
  if (tid == 0) {
    const float m = __builtin_fmaxf(__builtin_fmaxf(red[0], red[1]), __builtin_fmaxf(red[2], red[3]));
    kmax[int64_t(h) * n_kblk + b] = __builtin_sqrtf(m);
  }
}

}  // namespace

hipError_t launch_attn_fwd(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* o,
                           const int32_t* cu_seqlens, const float* slopes, float softmax_scale,
                           float* lse, float* kmax_ws, const g5moe_attn_shape& s,
                           hipStream_t st) {
  // Key-norm bounds: block skipping (with ALiBi) and the reference-max loop.  The
  // pre-pass is a launch and a read of k, 2-4 us for one sequence.  With the pass
  // against without, 12 heads, queries and keys N(0, 1), in brackets twice that (the
  // bounds then leave the online loop in place):
  //   ALiBi:  1 x 512 12.9, 11.0 (14.7, 11.1); 2 x 1,024 19.8, 19.4 (23.0, 19.6);
  //           8 x 1,024 43.6, 45.2 (49.2, 47.0); 1 x 4,550 57, 95 (81, 96)
  //   none:   1 x 512 11.9, 10.0 (13.7, 10.2); 4 x 1,536 52, 55 (58, 53);
  //           16 x 2,048 264, 286 (299, 288); 2 x 3,000 85, 93 (99, 94);
  //           8 x 4,550 594, 650 (674, 662)
  // So without ALiBi the scores, which the host cannot see, decide from about 1,500
  // tokens on; up to 2,048 the pass is left out.  With ALiBi the length of what is
  // skipped decides, and short calls keep the pass too: their outputs stay those of
  // the loop they always took.
  const bool bounds = kmax_ws != nullptr && s.total_tokens > 0 &&
                      (slopes != nullptr || s.max_seqlen > 2048);
  const int n_kblk = int((s.total_tokens + 63) / 64);
  if (bounds) {
    hipLaunchKernelGGL(key_norm_max_kernel, dim3(unsigned(n_kblk), unsigned(s.n_kv_heads)),
                       dim3(256), 0, st, k, s.k_token_stride, s.k_head_stride, s.total_tokens,
                       n_kblk, kmax_ws);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  AttnArgs a;
  a.q = q;
  a.k = k;
  a.v = v;
  a.o = o;
  a.cu_seqlens = cu_seqlens;
  a.q_tok = s.q_token_stride;
  a.k_tok = s.k_token_stride;
  a.v_tok = s.v_token_stride;
  a.o_tok = s.o_token_stride;
  a.q_head = s.q_head_stride;
  a.k_head = s.k_head_stride;
  a.v_head = s.v_head_stride;
  a.o_head = s.o_head_stride;
  a.group = s.n_heads / s.n_kv_heads;
  a.sc = softmax_scale * kLog2e;
  a.slopes = slopes;
  a.lse = lse;
  a.kmax = bounds ? kmax_ws : nullptr;
  a.n_kblk = n_kblk;
  a.total = s.total_tokens;
  const dim3 grid(unsigned((s.max_seqlen + kBQ - 1) / kBQ), unsigned(s.n_heads),
                  unsigned(s.n_seqs));
  // 64 rows of a k or v tile within 32-bit byte offsets
  const bool wide = std::max(s.k_token_stride, s.v_token_stride) >= (int64_t(1) << 24);
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, a); };
  const bool neg = softmax_scale < 0.0f;
  if (wide && lse != nullptr)
    neg ? launch(attn_fwd_kernel<true, true, true>) : launch(attn_fwd_kernel<true, true, false>);
  else if (wide)
    neg ? launch(attn_fwd_kernel<false, true, true>) : launch(attn_fwd_kernel<false, true, false>);
  else if (lse != nullptr)
    neg ? launch(attn_fwd_kernel<true, false, true>) : launch(attn_fwd_kernel<true, false, false>);
  else
    neg ? launch(attn_fwd_kernel<false, false, true>)
        : launch(attn_fwd_kernel<false, false, false>);
  return hipGetLastError();
}

}  // namespace g5moe
