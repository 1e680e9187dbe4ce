// Matrix-core tile pass at float32 fidelity for the two wrappers the reference names: pre-rotated scores over packed
// keys (tq_prerot_qk_scores) and the weighted value sum with given weights (tq_sparse_v_matvec), d = 128, 1 to 4 bits,
// n_rep <= 16.  Included by tq_attn.hip after tq_packed_mfma.h, whose layout it shares (a workgroup of 8 waves owns
// 512 positions of one kv head, a wave 64 of them).
//
// Every float32 operand enters as TWO fp16 numbers, its rounded value and the rounded remainder of that rounding
// (x = hi + lo to about 2^-22 |x|), and a product a * b is formed as hi_a hi_b + hi_a lo_b + lo_a hi_b: three
// v_mfma_f32_16x16x32_f16 per tile instead of one.  An fp16 x fp16 product has 22 significant bits and is exact in the
// float32 accumulator; what is dropped is lo_a lo_b, 2^-22 of the product.  So the result differs from a float32
// evaluation only by the order of the float32 additions: the reference's own bars for these two functions
// (1e-5 relative for the value sum, 1e-4 absolute for scores) hold with two orders of magnitude to spare, which the
// single-fp16 path (3e-4) does not meet.
//
//   centroids  scaled by 2^10 (exact) so that the remainders stay normal fp16 numbers; the pair table holds
//              {half2(hi, hi), half2(lo, lo)} per index: one 8-byte look-up per pair of elements;
//   queries    q_rot as hi / lo halves in LDS (as the fp16-operand pass already does);
//   weights    p = w * norm in float32 (the reference's order, (w * norm) * c), positions below the threshold
//              dropped, then scaled per wave by a power of two that puts the wave's largest p near 2^13 -- so that
//              weights many decades below the largest still have normal hi and lo parts -- and split.
//
// The composed decode step (pre-rotation, scores, softmax, thresholded value sum: tq_composed_decode) takes the same two passes
// as kSoftScores and kSoftWeights, for a batch: the query is rotated inside, the scores leave scaled and masked in log2 units
// with the statistics (maximum, sum of 2^(s - maximum)) of each tile, and the value pass makes the weights 2^(s - M) / L of the
// whole row itself.  As five operations (rotation, scores, a row softmax that reads every score eleven times, values, merge)
// plus a conversion and a copy, 28 / 4 heads over 65 536 positions took 60 us, of which the softmax 18; in three launches 31.
#pragma once

#include "tq_packed_mfma.h"

namespace tqm {

constexpr float kSplitTableScale = 1024.0f;
constexpr float kSplitTableUnscale = 1.0f / 1024.0f;

// this lane's entries of the split pair table: entry i = {half2(hi[i & mask], hi[i >> BITS]), half2(lo[..], lo[..])}
template <int BITS>
__device__ __forceinline__ void fill_split_table(uint2* lut, const Codebook& cb, int lane) {
  using VF = VField<BITS>;
#pragma unroll
  for (int base = 0; base < VF::kLut; base += 64) {
    const int idx = base + lane;
    float c0 = 0.0f, c1 = 0.0f;
#pragma unroll
    for (int i = 0; i < (1 << BITS); ++i) {
      c0 = ((idx & ((1 << BITS) - 1)) == i) ? cb.c[i] : c0;
      c1 = ((idx >> BITS) == i) ? cb.c[i] : c1;
    }
    c0 *= kSplitTableScale;
    c1 *= kSplitTableScale;
    const __half h0 = __float2half_rn(c0), h1 = __float2half_rn(c1);
    const uint32_t hi = pack_h2(__half2float(h0), __half2float(h1));
    const uint32_t lo = pack_h2(c0 - __half2float(h0), c1 - __half2float(h1));
    if (VF::kLut >= 64 || idx < VF::kLut) lut[idx] = make_uint2(hi, lo);
  }
}

struct SplitArgs {
  const float* q_rot;         // scores: [n_q, 128] f32, pre-rotated
  const void* q_raw;          // kSoftScores: [n_seq, n_q, 128] of q_dtype, rotated inside
  const float* k_signs;
  const float* mask;          // kSoftScores: additive rows or NULL
  float* stats;               // soft modes: [n_seq * n_kv, n_tiles, n_rep, 2]
  int64_t seq_stride, norms_seq_stride, mask_seq_stride, mask_head_stride;
  int32_t q_dtype;
  float scale2;               // kSoftScores: attention scale times log2 e
  const float* weights;       // values: [n_seq * n_q, w_stride] f32 weights; kSoftWeights: scores in log2 units
  int64_t w_stride;
  const uint32_t* packed;     // keys (scores) or values
  const float* norms;
  float* scores;              // scores: [n_q, seq_len] f32; kSoftScores: [n_seq * n_q, w_stride]
  float* ws_S;                // values: partial sums [n_kv, n_tiles, n_rep, 128]
  float* ws_ml;               //         their (0, sum of weights) pairs
  int64_t seq_len;
  int64_t head_stride, norms_head_stride;   // rows / floats between kv heads
  int32_t n_kv, n_rep, n_tiles;
  float scale;                // scores: 1 / dim
  float threshold;            // values
};

// MODE = kScores, kWeights: grid = (n_tiles, n_kv); kSoftScores, kSoftWeights: (n_tiles, n_kv, n_seq).  512 threads.
// F: tiles of scores or weights that share a register group (HeadLanes); keys wait in the registers that decode them (KeyQuarter).
// The composed step of 28 / 4 heads over 65 536 positions: scores 11.8 -> 10.8 us, values 14.0 -> 12.8.  With 32 copies of the
// look-up table, a lane's in banks of its own, 11.6 and 13.9: what the copies take to fill is more than the conflicts cost.
template <int MODE, int BITS, int F>
__global__ __launch_bounds__(kMfmaThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
void split_tile_kernel(SplitArgs a, Codebook cb) {
  using VF = VField<BITS>;
  using KQ = KeyQuarter<BITS>;
  using Lanes = HeadLanes<F>;
  constexpr int kGroups = Lanes::kGroups;
  constexpr int kPd = VF::kPd;
  constexpr bool SCORES = MODE == kScores || MODE == kSoftScores;
  constexpr bool SOFT_S = MODE == kSoftScores, SOFT_W = MODE == kSoftWeights;
  __shared__ __align__(16) unsigned char big_s[32768];      // per-wave 4 KB areas, later the merge deposits
  __shared__ __align__(16) uint2 lut_s[VF::kLut < 64 ? 64 : VF::kLut];
  __shared__ __align__(16) uint32_t q_s[kHeadsMax][kQPitch];
  __shared__ __align__(16) uint32_t ql_s[kHeadsMax][kQPitch];
  __shared__ __align__(16) float n_s[kWaves][kWavePos];
  __shared__ __align__(16) MergeLds<kWaves> mg_s;
  __shared__ float m_s[kWaves][kHeadsMax], l_s[kWaves][kHeadsMax];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15, g = lane >> 4;
  const int head = n16 % Lanes::kStep;                       // of the scores and weights in this lane's register groups
  const int first_pos = Lanes::row(0, n16, g);               // their first position in the wave's 64; group u is 16 F u further
  const int tile = blockIdx.x, kvh = blockIdx.y, seq = (SOFT_S || SOFT_W) ? blockIdx.z : 0;
  const int n_rep = a.n_rep;
  const int64_t grp = (int64_t)seq * a.n_kv + kvh;
  const int64_t q_row0 = grp * n_rep;
  const int64_t len = a.seq_len;
  const int64_t tile_p0 = (int64_t)tile * kTilePos;
  if (tile_p0 >= len) return;
  const int rows_here = (int)min((int64_t)kTilePos, len - tile_p0);
  const int last_row = rows_here - 1;
  const int wrow0 = wave * kWavePos;
  int crow = wrow0 + lane;
  crow = crow < last_row ? crow : last_row;

  // ---- loads ----------------------------------------------------------------------------------------------------
  float2 my_q[2];
  if (MODE == kScores) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int w = tid + i * kMfmaThreads;
      my_q[i] = (w < n_rep * (kD / 2)) ? reinterpret_cast<const float2*>(a.q_rot + q_row0 * kD)[w] : make_float2(0.f, 0.f);
    }
  }
  const int64_t seq_rows = (SOFT_S || SOFT_W) ? (int64_t)seq * a.seq_stride : 0;
  const float my_n = a.norms[((SOFT_S || SOFT_W) ? (int64_t)seq * a.norms_seq_stride : 0) + (int64_t)kvh * a.norms_head_stride + tile_p0 + crow];
  const uint32_t* block = a.packed + (seq_rows + (int64_t)kvh * a.head_stride + tile_p0 + wrow0) * kPd;
  PackedBlockT<kPd> blk;
  KQ kq[4];                                                  // keys: the lane's quarters of rows 16 t + n16, clamped into the tile
  if constexpr (SCORES) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
      kq[t].load_any(reinterpret_cast<const char*>(block - (int64_t)wrow0 * kPd), (uint32_t)min(wrow0 + 16 * t + n16, last_row) * (kPd * 4), g);
  } else {
    load_block(blk, block, lane, wrow0, rows_here);
  }
  // given weights: four positions of the lane's head per group
  float wgt[kGroups][4];
  if (!SCORES) {
    const bool vec_ok = ((a.w_stride & 3) == 0) && ((reinterpret_cast<uintptr_t>(a.weights) & 15) == 0);   // uniform
#pragma unroll
    for (int t = 0; t < kGroups; ++t) {
      const int row0 = wrow0 + 16 * F * t + first_pos;
      const float* src = a.weights + (q_row0 + head) * a.w_stride + tile_p0 + row0;
#pragma unroll
      for (int j = 0; j < 4; ++j) wgt[t][j] = SOFT_W ? -INFINITY : 0.0f;
      if (head < n_rep) {
        if (vec_ok && row0 + 4 <= rows_here) {
          const f4 v = *reinterpret_cast<const f4*>(src);
          wgt[t][0] = v[0]; wgt[t][1] = v[1]; wgt[t][2] = v[2]; wgt[t][3] = v[3];
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (row0 + j < rows_here) wgt[t][j] = src[j];
        }
      }
    }
  }
  // kSoftWeights: the statistics of the row's tiles, thread = head tid % 16, tiles tid / 16 + 32 u
  float M_part = -INFINITY, L_part = 0.0f;
  if (SOFT_W) {
    const float* st = a.stats + grp * a.n_tiles * (int64_t)(n_rep * 2);
    const int h = tid & 15;
    if (h < n_rep) {
      for (int t0 = tid >> 4; t0 < a.n_tiles; t0 += 128) {
        float2 ml[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          ml[u] = (t0 + 32 * u < a.n_tiles) ? *reinterpret_cast<const float2*>(st + (int64_t)(t0 + 32 * u) * (n_rep * 2) + 2 * h)
                                            : make_float2(-INFINITY, 0.0f);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float Mn = fmaxf(M_part, ml[u].x);
          L_part = (Mn == -INFINITY) ? L_part + ml[u].y                  // zeros, or the NaN of a tile without a number
                                     : L_part * __builtin_amdgcn_exp2f(M_part - Mn) + ml[u].y * __builtin_amdgcn_exp2f(ml[u].x - Mn);
          M_part = Mn;
        }
      }
    }
#pragma unroll
    for (int d = 16; d <= 32; d <<= 1) {
      const float Mo = shfl_xor_f(M_part, d), Lo = shfl_xor_f(L_part, d);
      const float Mn = fmaxf(M_part, Mo);
      L_part = (Mn == -INFINITY) ? L_part + Lo : L_part * __builtin_amdgcn_exp2f(M_part - Mn) + Lo * __builtin_amdgcn_exp2f(Mo - Mn);
      M_part = Mn;
    }
    if (lane < kHeadsMax) {
      m_s[wave][lane] = M_part;
      l_s[wave][lane] = L_part;
    }
  }
  if (tid < 64) fill_split_table<BITS>(lut_s, cb, tid);
  if (SOFT_S) rotate_query_rows<kWaves>(a.q_raw, a.q_dtype, a.k_signs, q_row0, n_rep, wave, lane, q_s, ql_s);
  if (MODE == kScores) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const __half2 h = __floats2half2_rn(my_q[i].x, my_q[i].y);
      const float2 back = __half22float2(h);
      (&q_s[0][0])[q_word(tid + i * kMfmaThreads)] = *reinterpret_cast<const uint32_t*>(&h);
      (&ql_s[0][0])[q_word(tid + i * kMfmaThreads)] = pack_h2(my_q[i].x - back.x, my_q[i].y - back.y);
    }
  }
  n_s[wave][lane] = SCORES ? my_n * (a.scale * kSplitTableUnscale) : my_n;
  __syncthreads();

  uint32_t* stage = reinterpret_cast<uint32_t*>(big_s) + wave * 1024;
  if constexpr (!SCORES) stage_block(blk, stage, lane);

  if constexpr (SCORES) {
    // ---- scores: A = centroids of 16 positions x 32 elements (hi, lo), B = query columns (hi, lo)
    u4 qreg[4], qlow[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
      for (int jp = 0; jp < 4; ++jp) {
        qreg[kb][jp] = q_s[n16][KQ::pair(kb, jp, g)];
        qlow[kb][jp] = ql_s[n16][KQ::pair(kb, jp, g)];
      }
    }
    typename Lanes::Group s[kGroups];
    const bool mask_vec = SOFT_S && a.mask && ((reinterpret_cast<uintptr_t>(a.mask) & 15) == 0) && ((a.mask_seq_stride & 3) == 0) &&
                          ((a.mask_head_stride & 3) == 0);                                         // uniform
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const uint32_t f = kq[t].field(kb, g);
        u4 kh, kl;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint2 e = lut_s[VF::index(f, k)];
          kh[k] = e.x;
          kl[k] = e.y;
        }
        // smallest terms first
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, kl), __builtin_bit_cast(h8, qreg[kb]), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, kh), __builtin_bit_cast(h8, qlow[kb]), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, kh), __builtin_bit_cast(h8, qreg[kb]), acc, 0, 0, 0);
      }
      Lanes::put(s, t, acc);
    }
#pragma unroll
    for (int t = 0; t < kGroups; ++t) {
      s[t] *= *reinterpret_cast<const f4*>(&n_s[wave][16 * F * t + first_pos]);
      if (SOFT_S) {
        const int row0 = wrow0 + 16 * F * t + first_pos;
        float mk[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (a.mask && head < n_rep)
          load_mask4(a.mask + (int64_t)seq * a.mask_seq_stride + ((int64_t)kvh * n_rep + head) * a.mask_head_stride + tile_p0 + row0,
                     row0, rows_here, mask_vec, mk);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float v = s[t][j] * a.scale2;
          s[t][j] = (row0 + j < rows_here) ? (a.mask ? __builtin_fmaf(mk[j], kLog2e, v) : v) : -INFINITY;
        }
      }
    }
    if (SOFT_S) {                                          // statistics of the lane's head over the wave's positions
      float m = -INFINITY, l = 0.0f;
#pragma unroll
      for (int t = 0; t < kGroups; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) m = fmaxf(m, s[t][j]);
      m = max_over_rows(Lanes::max_over_tiles(m));
      const float msafe = (m == -INFINITY) ? 0.0f : m;
#pragma unroll
      for (int t = 0; t < kGroups; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) l += __builtin_amdgcn_exp2f(s[t][j] - msafe);
      l = sum_over_rows(Lanes::sum_over_tiles(l));
      if (g == 0) {
        m_s[wave][n16] = m;
        l_s[wave][n16] = l;
      }
    }
    // The wave's 64 x n_rep scores leave through its LDS area (idle here: keys wait in registers): a store
    // instruction then writes whole 256-byte runs of a head's row.  Area = [16 heads][16 units of 4 positions],
    // the unit index xor-ed with the head (conflict-free 16-byte accesses both ways).
    f4* sc = reinterpret_cast<f4*>(stage);
#pragma unroll
    for (int t = 0; t < kGroups; ++t) sc[head * 16 + ((4 * F * t + first_pos / 4) ^ head)] = s[t];
    const int64_t row_len = SOFT_S ? a.w_stride : len;
    const bool vec_ok = ((row_len & 3) == 0) && ((reinterpret_cast<uintptr_t>(a.scores) & 15) == 0);   // uniform
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int h = 4 * i + g, unit = n16;
      if (h < n_rep) {
        const f4 v = sc[h * 16 + (unit ^ h)];
        const int row0 = wrow0 + 4 * unit;
        float* dst = a.scores + (q_row0 + h) * row_len + tile_p0 + row0;
        if (vec_ok && row0 + 4 <= rows_here) {
          __builtin_nontemporal_store(v, reinterpret_cast<f4*>(dst));     // streaming store: 10.9 -> 10.3 us at 65 536 positions
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (row0 + j < rows_here) dst[j] = v[j];
        }
      }
    }
    if (SOFT_S) {
      __syncthreads();
      if (tid < n_rep) {
        float M = m_s[0][tid], L = 0.0f;
#pragma unroll
        for (int w = 1; w < kWaves; ++w) M = fmaxf(M, m_s[w][tid]);
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          const float mw = m_s[w][tid];
          L += (mw == -INFINITY) ? l_s[w][tid] * 0.0f : l_s[w][tid] * __builtin_amdgcn_exp2f(mw - M);   // a NaN stays one
        }
        float* st = a.stats + (grp * a.n_tiles + tile) * (int64_t)(n_rep * 2);
        st[2 * tid] = M;
        st[2 * tid + 1] = L;
      }
    }
  } else {
    // ---- values: p = w * norm (weights below the threshold dropped), scaled per wave, split into hi and lo
    float p[kGroups][4];
    float pmax = 0.0f, l = 0.0f;
    if (SOFT_W) {                                          // the weight 2^(s - M) / L; a row without a visible position: 0 * inf = NaN,
      float M = -INFINITY, L = 0.0f;                       // as a softmax over nothing is
#pragma unroll
      for (int w = 0; w < kWaves; ++w) M = fmaxf(M, m_s[w][head]);
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const float mw = m_s[w][head];
        L += (mw == -INFINITY) ? l_s[w][head] * 0.0f : l_s[w][head] * __builtin_amdgcn_exp2f(mw - M);
      }
      if (M == -INFINITY) M = 0.0f;
      const float inv_l = 1.0f / L;
#pragma unroll
      for (int t = 0; t < kGroups; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          wgt[t][j] = (head < n_rep && wrow0 + 16 * F * t + first_pos + j < rows_here) ? __builtin_amdgcn_exp2f(wgt[t][j] - M) * inv_l : 0.0f;
    }
#pragma unroll
    for (int t = 0; t < kGroups; ++t) {
      const float4 n4 = *reinterpret_cast<const float4*>(&n_s[wave][16 * F * t + first_pos]);
      const float nv[4] = {n4.x, n4.y, n4.z, n4.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float w = (wgt[t][j] < a.threshold) ? 0.0f : wgt[t][j];
        l += w;
        p[t][j] = w * nv[j];
        pmax = fmaxf(pmax, fabsf(p[t][j]));
      }
    }
    pmax = wave_max(pmax);
    // 2^e with pmax * 2^e in [2^13, 2^14); exponents clamped so that both 2^e and 2^-e are normal floats
    int ex = (int)((__float_as_uint(pmax) >> 23) & 0xFF);                 // biased exponent of pmax (0: pmax is 0 or denormal)
    ex = ex < 40 ? (ex < 1 ? 140 : 40) : (ex > 230 ? 230 : ex);
    const float up = __uint_as_float((uint32_t)(254 - ex + 13) << 23);   // 2^(127 - ex + 13)
    const float inv_tscale = __uint_as_float((uint32_t)(ex - 13) << 23); // its inverse
    uint32_t pa_hi[2][4], pa_lo[2][4];
#pragma unroll
    for (int u = 0; u < kGroups; ++u) {
      float hi[4], lo[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float ps = p[u][j] * up;
        hi[j] = __half2float(__float2half_rn(ps));
        lo[j] = ps - hi[j];
      }
      const uint32_t h01 = pack_h2(hi[0], hi[1]), h23 = pack_h2(hi[2], hi[3]), l01 = pack_h2(lo[0], lo[1]), l23 = pack_h2(lo[2], lo[3]);
#pragma unroll
      for (int f = 0; f < F; ++f) {
        const int t = F * u + f;
        pa_hi[t >> 1][2 * (t & 1)] = Lanes::take(h01, f);
        pa_hi[t >> 1][2 * (t & 1) + 1] = Lanes::take(h23, f);
        pa_lo[t >> 1][2 * (t & 1)] = Lanes::take(l01, f);
        pa_lo[t >> 1][2 * (t & 1) + 1] = Lanes::take(l23, f);
      }
    }
    l = sum_over_rows(Lanes::sum_over_tiles(l));

    int w0, sh_lo, sh_hi;
    VF::pos(n16, w0, sh_lo, sh_hi);
    f4 accS[8];
#pragma unroll
    for (int et = 0; et < 8; ++et) accS[et] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb2 = 0; kb2 < 2; ++kb2) {
      uint32_t VI[8];
      value_indices<BITS, false>(stage, kb2, g, w0, sh_lo, sh_hi, VI);
      const u4 Ah = {pa_hi[kb2][0], pa_hi[kb2][1], pa_hi[kb2][2], pa_hi[kb2][3]};
      const u4 Al = {pa_lo[kb2][0], pa_lo[kb2][1], pa_lo[kb2][2], pa_lo[kb2][3]};
#pragma unroll
      for (int et = 0; et < 8; ++et) {
        u4 Bh, Bl;
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          const uint2 e = lut_s[VF::index(VI[(et & 1) * 4 + qd], et >> 1)];
          Bh[qd] = e.x;
          Bl[qd] = e.y;
        }
        accS[et] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, Al), __builtin_bit_cast(h8, Bh), accS[et], 0, 0, 0);
        accS[et] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, Ah), __builtin_bit_cast(h8, Bl), accS[et], 0, 0, 0);
        accS[et] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, Ah), __builtin_bit_cast(h8, Bh), accS[et], 0, 0, 0);
      }
    }
    float* pS = a.ws_S + (grp * a.n_tiles + tile) * (int64_t)(n_rep * kD);
    float* pml = a.ws_ml + (grp * a.n_tiles + tile) * (int64_t)(n_rep * 2);
    merge_waves<kWaves>(mg_s, big_s, 4096, accS, 0.0f, l, inv_tscale, kSplitTableUnscale, n_rep, pS, pml);
  }
}

template <int BITS>
void launch_split_tiles(int mode, dim3 grid, const SplitArgs& a, const Codebook& cb, hipStream_t stream) {
#define TQ_SPLIT(F_)                                                                                                    \
  do {                                                                                                                  \
    if (mode == kScores) split_tile_kernel<kScores, BITS, F_><<<grid, kMfmaThreads, 0, stream>>>(a, cb);                \
    else if (mode == kSoftScores) split_tile_kernel<kSoftScores, BITS, F_><<<grid, kMfmaThreads, 0, stream>>>(a, cb);   \
    else if (mode == kSoftWeights) split_tile_kernel<kSoftWeights, BITS, F_><<<grid, kMfmaThreads, 0, stream>>>(a, cb); \
    else split_tile_kernel<kWeights, BITS, F_><<<grid, kMfmaThreads, 0, stream>>>(a, cb);                               \
  } while (0)
  const int f = tiles_per_group(a.n_rep);
  if (f == 4) TQ_SPLIT(4);
  else if (f == 2) TQ_SPLIT(2);
  else TQ_SPLIT(1);
#undef TQ_SPLIT
}
#ifndef TQ_WIDTH_HERE
extern template void launch_split_tiles<1>(int, dim3, const SplitArgs&, const Codebook&, hipStream_t);
extern template void launch_split_tiles<2>(int, dim3, const SplitArgs&, const Codebook&, hipStream_t);
extern template void launch_split_tiles<4>(int, dim3, const SplitArgs&, const Codebook&, hipStream_t);
#endif

}  // namespace tqm
