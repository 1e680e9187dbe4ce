// Chunked-prefill attention over PACKED keys and values (d = 128, 1 to 4 bits) on the gfx950 matrix
// cores: a chunk of query rows (all q heads) against the packed cache up to the chunk's end,
// causal inside the chunk.  The reference has no kernel for this step: its prefill dequantises
// the whole cache to fp16 (cache.py:125-129, 209-210) and calls stock SDPA, i.e. it moves
// 256 B per cached vector where this path moves 56 B (at three bits) and never materialises K or V.
//
// Everything happens in the rotated domain, as in flash_attention.py:79-162:
//   q_rot = B(q * signs_K)                                  (one pass, rounded to fp16)
//   s[r, p] = <q_rot[r], c_K[idx_K[p]]> * norm_K[p] * attn_scale / d
//   O[r]    = sum_p softmax_p(s[r, .]) * norm_V[p] * c_V[idx_V[p]]
//   out[r]  = B(O[r]) * signs_V / d                         (one butterfly per output row)
// One launch for all sequences of a batch, query rotation and final butterfly included; where the key positions are
// split (few query rows against a long cache) a second one merges the splits and does the butterfly.
#include "tq_common.h"

#include <math.h>

namespace {

using namespace tqd;

typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int kD = 128;
constexpr int kBlkPos = 64;                     // key positions decoded into LDS per step
constexpr int kWaves = 8;
constexpr int kWaveRows = 32;                   // query rows per wavefront
constexpr int kThreads = kWaves * 64;
constexpr int kKStride = 136;                   // halfs per decoded key row in LDS (272 B: conflict-free b128 reads)
constexpr int kVStride = 72;                    // halfs per row of the transposed value block (144 B)
constexpr float kVnScale = 0.0625f;             // value norms enter the fp16 weights times 2^-4 (norms up to 1e6)
constexpr float kLog2e = 1.44269504088896340736f;
constexpr int kRowsPerWavePass = 16;            // four lanes per row in the merge kernel

struct PrefillArgs {
  const void* q;                // [n_seq, n_q, n_rows, 128] of q_dtype
  const float* k_signs;
  const float* v_signs;
  const uint32_t* k_packed;     // rows of a sequence and kv head at seq * k_seq_stride + kvh * k_head_stride
  const float* k_norms;
  const uint32_t* v_packed;
  const float* v_norms;
  void* out;                    // [n_seq, n_q, n_rows, 128] of out_dtype (one split)
  float* ws_O;                  // [n_splits, n_seq * n_q, n_rows, 128] unnormalised sums, rotated domain (several)
  float* ws_ml;                 // [n_splits, n_seq * n_q, n_rows, 2]   running maximum (log2 units), sum of weights
  int64_t n_rows, kv_len, q_pos0;
  int64_t k_seq_stride, kn_seq_stride, v_seq_stride, vn_seq_stride;
  int64_t k_head_stride, kn_head_stride, v_head_stride, vn_head_stride;
  int64_t split_len;            // multiple of kBlkPos
  int32_t n_seq, n_kv, n_rep, n_splits, n_row_wgs, causal;
  int32_t q_dtype, out_dtype, q_wide, out_wide;   // wide: 16-byte aligned
  float score_scale;            // attn_scale / d / key-table scale * log2(e)
  float unscale;                // 1 / d / the scales of values and norms
};

// butterfly stage between the lower and the upper 32 lanes of a wavefront
__device__ __forceinline__ float half_stage(float v, uint32_t flip) {
  typedef unsigned int u2_t __attribute__((ext_vector_type(2)));
  const u2_t r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1] ^ flip);        // lower: own + partner; upper: partner - own
}
__device__ __forceinline__ float max_of_halves(float v) {
  typedef unsigned int u2_t __attribute__((ext_vector_type(2)));
  const u2_t r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// elements at + 16 kb + j of the query as float32
__device__ __forceinline__ void load_query(const PrefillArgs& a, int64_t at, float (&x)[8][8]) {
  if (a.q_dtype == TQ_F32) {
    const float* src = reinterpret_cast<const float*>(a.q) + at;
    if (a.q_wide) {
#pragma unroll
      for (int kb = 0; kb < 8; ++kb) {
        const f4 lo = *reinterpret_cast<const f4*>(src + 16 * kb), hi = *reinterpret_cast<const f4*>(src + 16 * kb + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) { x[kb][j] = lo[j]; x[kb][4 + j] = hi[j]; }
      }
    } else {
#pragma unroll
      for (int kb = 0; kb < 8; ++kb)
#pragma unroll
        for (int j = 0; j < 8; ++j) x[kb][j] = src[16 * kb + j];
    }
    return;
  }
  const uint16_t* src = reinterpret_cast<const uint16_t*>(a.q) + at;
  u4 w[8];
  if (a.q_wide) {
#pragma unroll
    for (int kb = 0; kb < 8; ++kb) w[kb] = *reinterpret_cast<const u4*>(src + 16 * kb);
  } else {
#pragma unroll
    for (int kb = 0; kb < 8; ++kb)
#pragma unroll
      for (int j = 0; j < 4; ++j) w[kb][j] = src[16 * kb + 2 * j] | ((uint32_t)src[16 * kb + 2 * j + 1] << 16);
  }
  if (a.q_dtype == TQ_F16) {
#pragma unroll
    for (int kb = 0; kb < 8; ++kb)
#pragma unroll
      for (int j = 0; j < 8; ++j) x[kb][j] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[kb][j >> 1] >> (16 * (j & 1))));
  } else {
#pragma unroll
    for (int kb = 0; kb < 8; ++kb)
#pragma unroll
      for (int j = 0; j < 8; ++j) x[kb][j] = __uint_as_float((j & 1) ? w[kb][j >> 1] & 0xFFFF0000u : w[kb][j >> 1] << 16);
  }
}

template <typename TO>
__device__ __forceinline__ void store_out4(const PrefillArgs& a, int64_t at, const float (&x)[4]) {
  TO* dst = reinterpret_cast<TO*>(a.out) + at;
  if (a.out_wide) {
    struct __align__(4 * sizeof(TO)) Four { TO v[4]; } w;
#pragma unroll
    for (int j = 0; j < 4; ++j) store_from_float<TO>(&w.v[j], x[j]);
    *reinterpret_cast<Four*>(dst) = w;
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) store_from_float<TO>(dst + j, x[j]);
  }
}

// 512 threads: two wavefronts per SIMD, so that one's matrix instructions overlap the other's LDS reads and softmax
// arithmetic.  A wavefront owns 32 query rows of one head; the eight of a workgroup are consecutive in (row tile, head of the
// kv head), heads fastest, so that they share the decoded keys and values, a short prompt fills them, and under the causal rule
// a workgroup of grouped-query heads ends at the position of its own 32 to 64 rows instead of 256.  Workgroups are numbered
// with the kv head fastest (the XCDs serve different kv heads) and the last rows first: the longest start first.
// Per block of 64 key positions: all threads decode the packed rows (BITS bits per field) through centroid-pair tables into LDS
//   Ks[p][e]   keys, row-major, fp16
//   Vt[e][s]   values, transposed; position p = 16b + 8i + 4h + j sits in slot s = 16b + 8h + 4i + j,
//              the order in which the weights come out of the score accumulators
// then every wavefront runs S^T = K Q^T (MFMA 32x32x16, the query as fp16 value + fp16 remainder:
// rounding q_rot to one fp16 costs up to 1e-2 of an output row when an outlier channel of V
// cancels in the average), the online softmax on its accumulators, and O^T += V^T P^T with the
// accumulator registers of S^T reused as the B operand.  A lane holds ONE query row throughout (column of both products):
// 16 scores of a step per lane, one exchange between the wavefront's halves for the row's maximum, and factors that are
// the lane's own; with 16x16 tiles a row was spread over four lanes and the factors went through LDS.
// The packed words of the next block are fetched while the current one is computed.
// One split: the workgroup divides, does the butterfly (one exchange between halves, the rest in registers) and writes
// the output; else partial sums go to the workspace.
// What bounds it: the matrix cores are busy half of the time (1.65 TFLOP with the remainder against 131 072 positions and 512
// rows of 32 heads, 0.78 ms at the 2.1 PFLOP/s of a bare loop of these instructions), the vector unit as long; matrix
// instructions and operand reads alone take 1.19 ms, the decoding adds 0.13, the softmax 0.3.  512 rows of 32 heads at the end of
// 131 072 positions: 1.68 -> 1.60 ms a chunk (16x16 tiles, one head a workgroup, before); two prompts of 2 001 positions, 32 / 8 heads:
// 2 x (9 rotation + 117 + 19 merge) + 19 concatenation -> 125 us in one launch.
// QLO = false leaves the query remainder out (one matrix instruction per key operand instead of two): for callers
// that declare their data free of outlier channels.
template <int BITS, bool QLO = true>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void prefill_tile_kernel(PrefillArgs a, Codebook kcb, Codebook vcb) {
  using PF = PackedField<BITS>;
  constexpr int kPdim = PF::kPd;                    // words per packed row
  constexpr int kLut = PF::kLut < 64 ? 64 : PF::kLut;
  __shared__ __align__(16) _Float16 Ks2[2][kBlkPos * kKStride];
  __shared__ __align__(16) _Float16 Vt2[2][kD * kVStride];
  __shared__ uint32_t stK2[2][2 * kThreads + 4], stV2[2][2 * kThreads + 4];
  __shared__ __align__(16) float kn_s2[2][kBlkPos], vn_s2[2][kBlkPos];
  __shared__ uint32_t lutk_s[kLut], lutv_s[kLut];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n32 = lane & 31, hl = lane >> 5;
  uint32_t x = blockIdx.x;
  const int kvh = x % (uint32_t)a.n_kv;
  x /= (uint32_t)a.n_kv;
  const int seq = x % (uint32_t)a.n_seq;
  x /= (uint32_t)a.n_seq;
  const int split = x % (uint32_t)a.n_splits;
  const int wg = a.n_row_wgs - 1 - (int)(x / (uint32_t)a.n_splits);
  const int n_tiles = (int)((a.n_rows + kWaveRows - 1) / kWaveRows);
  const int wt = wg * kWaves + wave;
  const int row_tile = wt / a.n_rep;
  const int n_q = a.n_kv * a.n_rep;
  const int64_t head = (int64_t)seq * n_q + kvh * a.n_rep + (wt - row_tile * a.n_rep);
  const bool active = row_tile < n_tiles;                                // uniform over the wavefront
  const int64_t wrow0 = (int64_t)row_tile * kWaveRows;

  // key positions of this workgroup: its split, cut at the last position any of its rows may see
  const int64_t p_lo = (int64_t)split * a.split_len;
  int64_t p_hi = min(a.kv_len, p_lo + a.split_len);
  if (a.causal) {
    const int last_tile = min(n_tiles - 1, (wg * kWaves + kWaves - 1) / a.n_rep);
    p_hi = min(p_hi, a.q_pos0 + min(a.n_rows, ((int64_t)last_tile + 1) * kWaveRows));
  }

  if (tid < 64) PF::fill(lutk_s, kcb, tid);
  else if (tid < 128) PF::fill(lutv_s, vcb, tid - 64);

  // decode roles: keys -- position tid/8, chunks 2*(tid%8) and +1; values -- position pair tid%32, chunk tid/32.
  // Word offsets of the fields in a staged block, their shifts (the second word of a field of three bits: 30 less), and
  // where the decoded elements go: what a thread keeps through the loop.
  uint32_t kword[2], kshift[2], vword, vshift;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    int w0, lo, hi;
    PF::pos(2 * (tid & 7) + i, w0, lo, hi);
    kword[i] = (tid >> 3) * kPdim + w0;
    kshift[i] = lo;
  }
  {
    int w0, lo, hi;
    PF::pos(tid >> 5, w0, lo, hi);
    vword = 2 * (tid & 31) * kPdim + w0;
    vshift = lo;
  }
  const uint32_t kdst = (tid >> 3) * kKStride + 16 * (tid & 7);
  // slot of the even position p: p = 16b + 8i + 4h + j  ->  16b + 8h + 4i + j
  const uint32_t vp = 2 * (tid & 31);
  const uint32_t vdst = (tid >> 5) * 8 * kVStride + (vp & 48) + 8 * ((vp >> 2) & 1) + 4 * ((vp >> 3) & 1) + (vp & 3);

  const uint32_t* kbase = a.k_packed + ((int64_t)seq * a.k_seq_stride + (int64_t)kvh * a.k_head_stride) * kPdim;
  const uint32_t* vbase = a.v_packed + ((int64_t)seq * a.v_seq_stride + (int64_t)kvh * a.v_head_stride) * kPdim;
  const float* knbase = a.k_norms + (int64_t)seq * a.kn_seq_stride + (int64_t)kvh * a.kn_head_stride;
  const float* vnbase = a.v_norms + (int64_t)seq * a.vn_seq_stride + (int64_t)kvh * a.vn_head_stride;
  const float* nbase = wave == 0 ? knbase : vnbase;                      // wavefronts 0 and 1 bring the norms

  // Packed words and norms of a block, without a branch: bases the same for the wavefront, 32-bit offsets, and what lies
  // past the end is fetched from the last word or norm that exists (real data of a row whose weights are zero).
  uint32_t pk[2], pv[2];
  float pn = 0.0f, pn_staged = 0.0f;
  auto prefetch = [&](int64_t pb) {
    const uint32_t rows = (uint32_t)min((int64_t)kBlkPos, a.kv_len - pb);
    const uint32_t last = rows * kPdim - 1;
    const uint32_t* kblk = kbase + pb * kPdim;
    const uint32_t* vblk = vbase + pb * kPdim;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t id = min((uint32_t)(tid + kThreads * i), last);
      pk[i] = kblk[id];
      pv[i] = vblk[id];
    }
    pn = (nbase + pb)[min((uint32_t)lane, rows - 1)];
  };

  if (p_lo < p_hi) prefetch(p_lo);

  // ---- query operands: B[k = element][n = row], lane (row n32, half hl) holds elements 16 kb + 8 hl + j: the rotated row
  // B(q * signs_K) as fp16 value and fp16 remainder of that rounding
  u4 qhi[8], qlo[8];
  {
    const int64_t r = wrow0 + n32;
    const bool ok = active && r < a.n_rows;
    const int64_t at = (head * a.n_rows + r) * kD;
    const uint32_t flip = hl ? 0x80000000u : 0u;
    float xs[8][8];
#pragma unroll
    for (int kb = 0; kb < 8; ++kb)
#pragma unroll
      for (int j = 0; j < 8; ++j) xs[kb][j] = 0.0f;
    if (ok) load_query(a, at + 8 * hl, xs);
#pragma unroll
    for (int kb = 0; kb < 8; ++kb) {
#pragma unroll
      for (int j = 0; j < 8; ++j) xs[kb][j] *= a.k_signs[16 * kb + 8 * hl + j];
#pragma unroll
      for (int h = 1; h < 8; h <<= 1)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (!(j & h)) {
            const float u = xs[kb][j], v = xs[kb][j + h];
            xs[kb][j] = u + v;
            xs[kb][j + h] = u - v;
          }
#pragma unroll
      for (int j = 0; j < 8; ++j) xs[kb][j] = half_stage(xs[kb][j], flip);
    }
#pragma unroll
    for (int h = 1; h < 8; h <<= 1)
#pragma unroll
      for (int kb = 0; kb < 8; ++kb)
        if (!(kb & h)) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float u = xs[kb][j], v = xs[kb + h][j];
            xs[kb][j] = u + v;
            xs[kb + h][j] = u - v;
          }
        }
#pragma unroll
    for (int kb = 0; kb < 8; ++kb)
#pragma unroll
      for (int jp = 0; jp < 4; ++jp) {
        const __half2 h = __floats2half2_rn(xs[kb][2 * jp], xs[kb][2 * jp + 1]);
        const float2 back = __half22float2(h);
        qhi[kb][jp] = *reinterpret_cast<const uint32_t*>(&h);
        qlo[kb][jp] = pack_h2(xs[kb][2 * jp] - back.x, xs[kb][2 * jp + 1] - back.y);
      }
  }

  f16v oacc[4];                                                          // O^T: elements 32 et + 8 (i / 4) + 4 hl + i % 4 of row n32
#pragma unroll
  for (int et = 0; et < 4; ++et)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[et][i] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;                                 // of row n32; l_run over the positions of this half
  // positions below which the wavefront's last row sees
  const int64_t last_lim = !active ? 0 : a.causal ? min(a.kv_len, a.q_pos0 + min(a.n_rows, wrow0 + kWaveRows)) : a.kv_len;

  // Pipeline over blocks with ONE barrier per block: block b+1 is decoded into the other LDS
  // buffer in the same stretch of code that computes block b.
  auto stage = [&](int sb) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      stK2[sb][tid + kThreads * i] = pk[i];
      stV2[sb][tid + kThreads * i] = pv[i];
    }
    pn_staged = pn;
  };
  // Decoding of a staged block in six steps: words, key look-ups, value look-ups, norms, key rows, value rows (transposed).
  struct Decode { uint32_t k[2][2], v[2][2]; u4 kw[2]; uint32_t vw[8]; };
  auto decode_step = [&](Decode& d, int sb, int step) {
    if (step == 0) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int w = 0; w < (BITS == 3 ? 2 : 1); ++w) {
          d.k[i][w] = stK2[sb][kword[i] + w];
          d.v[i][w] = stV2[sb][vword + i * kPdim + w];
        }
    } else if (step == 1) {                                              // keys: 16 elements of one position
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t f = PF::field(d.k[i], kshift[i], 30 - kshift[i]);
#pragma unroll
        for (int jp = 0; jp < 4; ++jp) d.kw[i][jp] = lutk_s[PF::index(f, jp)];
      }
    } else if (step == 2) {                                              // values: two positions x 8 elements
      uint32_t X, Y;                                                     // elements 8c + 0, 2, 4, 6 / 8c + 1, 3, 5, 7
      PF::interleave(PF::field(d.v[0], vshift, 30 - vshift), PF::field(d.v[1], vshift, 30 - vshift), X, Y);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        d.vw[2 * i] = lutv_s[PF::index(X, i)];
        d.vw[2 * i + 1] = lutv_s[PF::index(Y, i)];
      }
    } else if (step == 3) {
      if (wave == 0) kn_s2[sb][lane] = pn_staged * a.score_scale;
      else if (wave == 1) vn_s2[sb][lane] = pn_staged * kVnScale;
    } else if (step == 4) {
#pragma unroll
      for (int i = 0; i < 2; ++i) *reinterpret_cast<u4*>(&Ks2[sb][kdst + 8 * i]) = d.kw[i];
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) *reinterpret_cast<uint32_t*>(&Vt2[sb][vdst + i * kVStride]) = d.vw[i];
    }
  };
  auto decode = [&](int sb) {
    Decode d;
#pragma unroll
    for (int step = 0; step < 6; ++step) decode_step(d, sb, step);
  };
  // ---- pieces of a block's work, on sub-blocks h of 32 positions.  Scores S^T = K Q^T: register i of the accumulator is position
  // 32h + 8 (i / 4) + 4 hl + i % 4 of row n32.  Online softmax of the lane's row in eight steps, which leave the weights times
  // value norms as the B operand of the value product (P^T: slots 16 ks + 8 hl + j) and the factor of the sums so far.
  struct Soft { f16v s; f4 n0, n1; float mx, msafe, alpha, lsum; u4 P[2]; };
  auto k_operand = [&](int sb, int h, int kb) {
    return *reinterpret_cast<const u4*>(Ks2[sb] + (32 * h + n32) * kKStride + 8 * hl + 16 * kb);
  };
  auto v_operand = [&](int sb, int h, int i) {                           // i = 4 ks + et
    return *reinterpret_cast<const u4*>(Vt2[sb] + (32 * (i & 3) + n32) * kVStride + 8 * hl + 32 * h + 16 * (i >> 2));
  };
  auto norms4 = [&](const float* n, int h, int qd) { return *reinterpret_cast<const f4*>(n + 32 * h + 4 * hl + 8 * qd); };
  auto score_step = [&](f16v& s, const u4& k, int kb) {
    const h8 A = __builtin_bit_cast(h8, k);
    if (QLO) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(A, __builtin_bit_cast(h8, qlo[kb]), s, 0, 0, 0);
    s = __builtin_amdgcn_mfma_f32_32x32x16_f16(A, __builtin_bit_cast(h8, qhi[kb]), s, 0, 0, 0);
  };
  auto value_step = [&](const Soft& f, const u4& v, int i) {
    oacc[i & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, v), __builtin_bit_cast(h8, f.P[i >> 2]), oacc[i & 3], 0, 0, 0);
  };
  auto soft_start = [&](Soft& f, int sb, int h) {
    f.n0 = norms4(kn_s2[sb], h, 0);
    f.n1 = norms4(kn_s2[sb], h, 1);
  };
  auto soft_step = [&](Soft& f, int sb, int h, int step) {
    if (step < 2) {                                                      // scale by key norm (log2 units)
#pragma unroll
      for (int j = 0; j < 4; ++j) { f.s[8 * step + j] *= f.n0[j]; f.s[8 * step + 4 + j] *= f.n1[j]; }
      if (step == 0) {
        f.n0 = norms4(kn_s2[sb], h, 2);
        f.n1 = norms4(kn_s2[sb], h, 3);
      }
    } else if (step == 2) {
      f.mx = f.s[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) f.mx = fmaxf(f.mx, f.s[i]);
      f.n0 = norms4(vn_s2[sb], h, 0);
    } else if (step == 3) {
      const float m_new = fmaxf(m_run, max_of_halves(f.mx));
      f.msafe = (m_new == -INFINITY) ? 0.0f : m_new;
      f.alpha = __builtin_amdgcn_exp2f(m_run - f.msafe);                 // v_exp_f32: 2^-inf = 0, tiny results flush to 0
      m_run = m_new;
      f.lsum = 0.0f;
      f.n1 = norms4(vn_s2[sb], h, 1);
    } else {
      const int qd = step - 4;
      f4& vn = (qd & 1) ? f.n1 : f.n0;
      float p[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        p[j] = __builtin_amdgcn_exp2f(f.s[4 * qd + j] - f.msafe);
        f.lsum += p[j];
      }
      f.P[qd >> 1][2 * (qd & 1)] = pack_h2(p[0] * vn[0], p[1] * vn[1]);
      f.P[qd >> 1][2 * (qd & 1) + 1] = pack_h2(p[2] * vn[2], p[3] * vn[3]);
      asm volatile("" : "+v"(f.P[qd >> 1][2 * (qd & 1)]), "+v"(f.P[qd >> 1][2 * (qd & 1) + 1]), "+v"(f.lsum));   // computed here, not after the branch of the rescaling
      if (qd < 2) vn = norms4(vn_s2[sb], h, qd + 2);
      if (qd == 3) l_run = l_run * f.alpha + f.lsum;
    }
  };
  auto rescale = [&](float alpha) {                                      // when some running maximum moved
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int et = 0; et < 4; ++et)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[et][i] *= alpha;
    }
  };
  auto clear = [](f16v& s) {
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.0f;
  };
  auto compute_full = [&](int sb) {
      // Every row sees the whole block.  The matrix instructions alternate with steps of the vector work that does not
      // depend on them -- the decoding of the next block under the scores of sub-block 0, the softmax of sub-block 0 under the scores of
      // sub-block 1, the softmax of sub-block 1 under the values of both -- so that the matrix cores run while the vector unit
      // does; operands come two steps ahead, the fences keep the order.
      Soft f0, f1;
      Decode d;
      u4 op[3];
      clear(f0.s);
      op[0] = k_operand(sb, 0, 0);
      op[1] = k_operand(sb, 0, 1);
      decode_step(d, sb ^ 1, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kb = 0; kb < 8; ++kb) {
        if (kb + 2 < 8) op[(kb + 2) % 3] = k_operand(sb, 0, kb + 2);
        score_step(f0.s, op[kb % 3], kb);
        if (kb == 1) decode_step(d, sb ^ 1, 1);
        if (kb == 2) decode_step(d, sb ^ 1, 2);
        if (kb == 4) decode_step(d, sb ^ 1, 4);
        if (kb == 5) decode_step(d, sb ^ 1, 5);
        __builtin_amdgcn_sched_barrier(0);
      }
      clear(f1.s);
      soft_start(f0, sb, 0);
      op[0] = k_operand(sb, 1, 0);
      op[1] = k_operand(sb, 1, 1);
      decode_step(d, sb ^ 1, 3);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kb = 0; kb < 8; ++kb) {
        if (kb + 2 < 8) op[(kb + 2) % 3] = k_operand(sb, 1, kb + 2);
        score_step(f1.s, op[kb % 3], kb);
        soft_step(f0, sb, 0, kb);
        __builtin_amdgcn_sched_barrier(0);
      }
      rescale(f0.alpha);
      soft_start(f1, sb, 1);
      op[0] = v_operand(sb, 0, 0);
      op[1] = v_operand(sb, 0, 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        op[(i + 2) % 3] = v_operand(sb, (i + 2) >> 3, (i + 2) & 7);
        value_step(f0, op[i % 3], i);
        if (i < 6) soft_step(f1, sb, 1, i);
        __builtin_amdgcn_sched_barrier(0);
      }
      rescale(f1.alpha);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (i + 2 < 8) op[(i + 10) % 3] = v_operand(sb, 1, i + 2);
        value_step(f1, op[(i + 8) % 3], i);
        if (i == 0) soft_step(f1, sb, 1, 6);
        if (i == 2) soft_step(f1, sb, 1, 7);
        __builtin_amdgcn_sched_barrier(0);
      }
  };
  auto compute_edge = [&](int sb, int64_t pb) {
    {
      // the lane's row sees positions below lim, sub-block 0 its own positions 8 qd + j below rel
      const int64_t left = min(a.kv_len - pb, (int64_t)kBlkPos);
      const int lim = a.causal ? (int)min(left, max((int64_t)-kBlkPos, a.q_pos0 + wrow0 + 1 - pb) + n32) : (int)left;
      const int rel = lim - 4 * hl;
#pragma nounroll
      for (int h = 0; h < 2; ++h) {
        if (pb + 32 * h >= last_lim) break;                              // no row of this wavefront sees the sub-block
        Soft f;
        clear(f.s);
#pragma unroll
        for (int kb = 0; kb < 8; ++kb) score_step(f.s, k_operand(sb, h, kb), kb);
        soft_start(f, sb, h);
#pragma unroll
        for (int step = 0; step < 8; ++step) {
          if (step == 2) {                                               // own positions 8 qd + j are visible below rel - 32 h
#pragma unroll
            for (int i = 0; i < 16; ++i) f.s[i] = (8 * (i >> 2) + (i & 3) >= rel - 32 * h) ? -INFINITY : f.s[i];
          }
          soft_step(f, sb, h, step);
        }
        rescale(f.alpha);
#pragma unroll
        for (int i = 0; i < 8; ++i) value_step(f, v_operand(sb, h, i), i);
      }
    }
  };

  if (p_lo < p_hi) {
    stage(0);
    __syncthreads();
    if (p_lo + kBlkPos < p_hi) prefetch(p_lo + kBlkPos);
    decode(0);
  }
  // positions that every row of the workgroup sees: blocks without a mask
  const int64_t wg_full = a.causal ? min(a.kv_len, a.q_pos0 + (int64_t)(wg * kWaves / a.n_rep) * kWaveRows + 1) : a.kv_len;
  int sb = 0;
  int64_t pb = p_lo;
  auto advance = [&]() {
    const bool more = pb + kBlkPos < p_hi;
    if (more) stage(sb ^ 1);               // words of block b+1 (fetched during block b-1)
    __syncthreads();                       // block b decoded by all; block b-1 computed by all; stage of b+1 visible
    if (pb + 2 * kBlkPos < p_hi) prefetch(pb + 2 * kBlkPos);
    return more;
  };
  for (; pb < p_hi && pb + kBlkPos <= wg_full; pb += kBlkPos, sb ^= 1) {
    advance();
    compute_full(sb);                      // decodes block b+1, or, after the last one, what is staged, for nobody
  }
  for (; pb < p_hi; pb += kBlkPos, sb ^= 1) {
    if (advance()) decode(sb ^ 1);
    compute_edge(sb, pb);
  }

  const int64_t r = wrow0 + n32;
  if (!active || r >= a.n_rows) return;
  float l;
  {
    typedef unsigned int u2_t __attribute__((ext_vector_type(2)));
    const u2_t w = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run), __float_as_uint(l_run), false, false);
    l = __uint_as_float(w[0]) + __uint_as_float(w[1]);
  }
  if (a.n_splits > 1) {
    // ---- partial results of this split
    const int64_t part = ((int64_t)split * a.n_seq * n_q + head) * a.n_rows + r;
    if (hl == 0) {
      a.ws_ml[part * 2] = m_run;
      a.ws_ml[part * 2 + 1] = l;
    }
    float* orow = a.ws_O + part * kD + 4 * hl;
#pragma unroll
    for (int et = 0; et < 4; ++et)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd)
        *reinterpret_cast<f4*>(orow + 32 * et + 8 * qd) =
            f4{oacc[et][4 * qd], oacc[et][4 * qd + 1], oacc[et][4 * qd + 2], oacc[et][4 * qd + 3]};
    return;
  }
  if (m_run == -INFINITY) {                                              // none of the row's scores was a number: zeros, as in the
#pragma unroll                                                           // merge of several splits
    for (int et = 0; et < 4; ++et)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[et][i] = 0.0f;
  }
  // ---- out[r] = B(O[r]) * signs_V * unscale / l : strides 1, 2 (registers), 4 (halves), 8, 16 and 32, 64 (registers)
  const uint32_t flip = hl ? 0x80000000u : 0u;
#pragma unroll
  for (int et = 0; et < 4; ++et) {
#pragma unroll
    for (int h = 1; h < 4; h <<= 1)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (!(i & h)) {
          const float u = oacc[et][i], v = oacc[et][i + h];
          oacc[et][i] = u + v;
          oacc[et][i + h] = u - v;
        }
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[et][i] = half_stage(oacc[et][i], flip);
#pragma unroll
    for (int h = 4; h < 16; h <<= 1)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (!(i & h)) {
          const float u = oacc[et][i], v = oacc[et][i + h];
          oacc[et][i] = u + v;
          oacc[et][i + h] = u - v;
        }
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float a0 = oacc[0][i] + oacc[1][i], a1 = oacc[0][i] - oacc[1][i];
    const float a2 = oacc[2][i] + oacc[3][i], a3 = oacc[2][i] - oacc[3][i];
    oacc[0][i] = a0 + a2; oacc[2][i] = a0 - a2;
    oacc[1][i] = a1 + a3; oacc[3][i] = a1 - a3;
  }
  const float scale = (l > 0.0f) ? a.unscale / l : 0.0f;
  const int64_t at = (head * a.n_rows + r) * kD + 4 * hl;
#pragma unroll
  for (int et = 0; et < 4; ++et)
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
      float y[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = oacc[et][4 * qd + j] * a.v_signs[32 * et + 8 * qd + 4 * hl + j] * scale;
      const int64_t o = at + 32 * et + 8 * qd;
      if (a.out_dtype == TQ_F32) store_out4<float>(a, o, y);
      else if (a.out_dtype == TQ_F16) store_out4<__half>(a, o, y);
      else store_out4<__hip_bfloat16>(a, o, y);
    }
}

// Merge of the splits and the final butterfly: out[r] = B(sum_s f_s O_s[r]) * signs_V * unscale / L,
// f_s = 2^(m_s - max m), L = sum_s f_s l_s.  Four lanes per row.
template <typename TO>
__global__ __launch_bounds__(256) void prefill_merge_kernel(const float* __restrict__ ws_O,
                                                            const float* __restrict__ ws_ml,
                                                            const float* __restrict__ signs, TO* __restrict__ out,
                                                            int64_t n /* n_q * n_rows */, int n_splits, float unscale) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int ls = lane & 3, v = lane >> 2;
  const int64_t row = ((int64_t)blockIdx.x * 4 + (tid >> 6)) * kRowsPerWavePass + v;
  const bool ok = row < n;
  const int64_t rr = ok ? row : 0;
  float M = -INFINITY;
  for (int s = 0; s < n_splits; ++s) M = fmaxf(M, ws_ml[((int64_t)s * n + rr) * 2]);
  float acc[4][8];
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[k][j] = 0.0f;
  float L = 0.0f;
  for (int s = 0; s < n_splits; ++s) {
    const float ms = ws_ml[((int64_t)s * n + rr) * 2];
    if (ms == -INFINITY) continue;                                       // this split saw no position of the row
    const float f = exp2f(ms - M);
    L += f * ws_ml[((int64_t)s * n + rr) * 2 + 1];
    const float* src = ws_O + ((int64_t)s * n + rr) * kD + 8 * ls;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float4 x0 = *reinterpret_cast<const float4*>(src + 32 * k);
      const float4 x1 = *reinterpret_cast<const float4*>(src + 32 * k + 4);
      acc[k][0] += f * x0.x; acc[k][1] += f * x0.y; acc[k][2] += f * x0.z; acc[k][3] += f * x0.w;
      acc[k][4] += f * x1.x; acc[k][5] += f * x1.y; acc[k][6] += f * x1.z; acc[k][7] += f * x1.w;
    }
  }
  butterfly_4lane(acc, (ls & 1) ? 0x80000000u : 0u, (ls & 2) ? 0x80000000u : 0u);
  const float scale = (L > 0.0f) ? unscale / L : 0.0f;
  if (ok) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int e = 32 * k + 8 * ls + j;
        store_from_float<TO>(out + row * kD + e, acc[k][j] * signs[e] * scale);
      }
  }
}

struct SplitPlan { int n_splits; int64_t split_len; };

// Workgroups per (sequence, kv head): eight wavefronts of 32 rows of one head each.
int64_t row_workgroups(int n_rep, int64_t n_rows) {
  return ((n_rows + kWaveRows - 1) / kWaveRows * n_rep + kWaves - 1) / kWaves;
}

// Splits of the key positions.  A workgroup fills a CU (LDS), so 256 run at once; a block of 64 positions takes one about
// 3.5 us, and more than one split costs a merge: the partial sums once out and once in (1 KB per row and split, about 4 TB/s) and
// a launch.  Estimated in blocks, smallest count within 3 % of the best:
//  - workgroups of about the same length (a chunk at the end of a long cache): rounds of 256 times the blocks of a split;
//  - of different lengths (a prompt under the causal rule, longest first): the even share of all blocks, at least the
//    longest workgroup.
// At least 8 blocks of positions per split, at most 32 splits, and never more than `fit`.  A plan is a function of the shape
// alone, never of the bytes at hand: results of equal calls are equal whatever ran before.
SplitPlan plan_splits(int n_seq, int n_kv, int n_rep, int64_t n_rows, int64_t kv_len, int64_t q_pos0, bool causal, int64_t fit) {
  const int64_t blocks = (kv_len + kBlkPos - 1) / kBlkPos;
  const int64_t wgs = row_workgroups(n_rep, n_rows), cols = wgs * n_kv * n_seq;
  const double merge_per_split = (double)n_seq * n_kv * n_rep * (double)n_rows * 1024.0 / 4e6 / 3.5;
  // blocks that the first and the last rows see; in between they grow evenly
  const int64_t first = causal ? (q_pos0 + 1 + kBlkPos - 1) / kBlkPos : blocks;
  const bool even = first * 5 >= blocks * 4;
  const double share = (double)cols * (double)(first + blocks) / 2.0 / 256.0 * 1.05;
  int64_t most = blocks / 8 > 0 ? blocks / 8 : 1;
  if (most > 32) most = 32;
  if (most > fit) most = fit > 0 ? fit : 1;
  int64_t want = 1;
  double best = 1e30;
  for (int64_t n = 1; n <= most; ++n) {
    const double longest = (double)((blocks + n - 1) / n);
    double cost = even ? (double)((cols * n + 255) / 256) * longest : (share > longest ? share : longest);
    if (n > 1) cost += merge_per_split * (double)n + 1.5;
    if (cost < best * 0.97) { best = cost; want = n; }
  }
  const int64_t per = (blocks + want - 1) / want;
  SplitPlan p;
  p.split_len = per * kBlkPos;
  p.n_splits = (int)((blocks + per - 1) / per);
  if (p.n_splits < 1) p.n_splits = 1;
  return p;
}

size_t align256(size_t v) { return (v + 255) / 256 * 256; }

size_t workspace_of(int64_t n_splits, size_t rows) {
  return n_splits <= 1 ? 0 : align256((size_t)n_splits * rows * kD * sizeof(float)) + align256((size_t)n_splits * rows * 2 * sizeof(float));
}

int64_t visible(int64_t kv_len, int64_t q_pos0, int64_t n_rows, bool causal) {
  return causal && q_pos0 + n_rows < kv_len ? q_pos0 + n_rows : kv_len;   // past the last row's own no position is seen
}

struct PrefillCall {
  const void* q; int q_dtype;
  const uint32_t* k_packed; const float* k_norms; const uint32_t* v_packed; const float* v_norms;
  const float* k_centroids; const float* v_centroids; const float* k_signs; const float* v_signs;
  void* out; int out_dtype;
  void* workspace; size_t workspace_bytes;
  int n_seq, n_kv_heads, n_rep;
  int64_t n_rows, kv_len, q_pos0;
  int64_t k_seq_stride, kn_seq_stride, v_seq_stride, vn_seq_stride;
  int64_t k_head_stride, kn_head_stride, v_head_stride, vn_head_stride;
  int dim, bits;
  float attn_scale;
  int flags;
  hipStream_t stream;
};

// `need`: the workspace that the entry point asks its callers for; `most`: the splits that it has room for
int prefill(const char* who, const PrefillCall& c, size_t need, int64_t most) {
  if (c.flags & ~(TQ_PREFILL_CAUSAL | TQ_PREFILL_FP16_QUERY))
    return tq::fail(TQ_ERR_ARG, "%s: unknown flag bits 0x%x", who, c.flags);
  const bool causal = c.flags & TQ_PREFILL_CAUSAL;
  if (int rc = tq::check_dim_bits(c.dim, c.bits)) return rc;
  if (c.dim != kD)
    return tq::fail(TQ_ERR_UNSUPPORTED, "%s: only dim 128 has a kernel, got dim %d", who, c.dim);
  if (c.n_seq < 1) return tq::fail(TQ_ERR_ARG, "%s: n_seq must be >= 1, got %d", who, c.n_seq);
  if (c.n_kv_heads < 1) return tq::fail(TQ_ERR_ARG, "%s: n_kv_heads must be >= 1, got %d", who, c.n_kv_heads);
  if (c.n_rep < 1) return tq::fail(TQ_ERR_NREP, "%s: n_rep must be >= 1, got %d", who, c.n_rep);
  if (tq::check_dtype(c.q_dtype) || tq::check_dtype(c.out_dtype)) return tq::fail(TQ_ERR_DTYPE, "%s: unknown dtype", who);
  if (c.n_rows < 0 || c.kv_len < 0 || c.q_pos0 < 0) return tq::fail(TQ_ERR_ARG, "%s: negative size", who);
  if (c.n_rows == 0) return TQ_OK;
  if (c.kv_len < 1) return tq::fail(TQ_ERR_ARG, "%s: kv_len must be >= 1", who);
  if (causal && c.q_pos0 + 1 > c.kv_len)
    return tq::fail(TQ_ERR_ARG, "%s: causal chunk starts at position %lld beyond the %lld cached positions", who,
                    (long long)c.q_pos0, (long long)c.kv_len);
  if (c.k_head_stride < c.kv_len || c.kn_head_stride < c.kv_len || c.v_head_stride < c.kv_len || c.vn_head_stride < c.kv_len)
    return tq::fail(TQ_ERR_ARG, "%s: a head stride is smaller than kv_len (%lld)", who, (long long)c.kv_len);
  if (!c.q || !c.k_packed || !c.k_norms || !c.v_packed || !c.v_norms || !c.k_centroids || !c.v_centroids || !c.k_signs ||
      !c.v_signs || !c.out || !c.workspace)
    return tq::fail(TQ_ERR_NULL, "%s: null pointer", who);
  if (!tq::aligned(c.q, tq::dtype_size(c.q_dtype)) || !tq::aligned(c.out, tq::dtype_size(c.out_dtype)) ||
      !tq::aligned(c.k_packed, 4) || !tq::aligned(c.v_packed, 4) || !tq::aligned(c.workspace, 256))
    return tq::fail(TQ_ERR_ALIGN, "%s: misaligned pointer (workspace needs 256 bytes)", who);
  if (c.workspace_bytes < need)
    return tq::fail(TQ_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who, need, c.workspace_bytes);
  const int n_q = c.n_kv_heads * c.n_rep;
  const size_t rows = (size_t)c.n_seq * n_q * (size_t)c.n_rows;
  const int64_t kv_eff = visible(c.kv_len, c.q_pos0, c.n_rows, causal);
  const SplitPlan plan = plan_splits(c.n_seq, c.n_kv_heads, c.n_rep, c.n_rows, kv_eff, c.q_pos0, causal, most);
  const int64_t row_wgs = row_workgroups(c.n_rep, c.n_rows);
  const int64_t grid = row_wgs * plan.n_splits * c.n_seq * c.n_kv_heads;
  if (grid >= (int64_t)1 << 31) return tq::fail(TQ_ERR_ARG, "%s: %lld query rows are too many", who, (long long)c.n_rows);

  PrefillArgs a{};
  a.q = c.q; a.k_signs = c.k_signs; a.v_signs = c.v_signs;
  a.k_packed = c.k_packed; a.v_packed = c.v_packed; a.k_norms = c.k_norms; a.v_norms = c.v_norms;
  a.out = c.out;
  a.ws_O = (float*)c.workspace;
  a.ws_ml = (float*)((char*)c.workspace + align256((size_t)plan.n_splits * rows * kD * sizeof(float)));
  a.n_rows = c.n_rows; a.kv_len = kv_eff; a.q_pos0 = c.q_pos0;
  a.k_seq_stride = c.k_seq_stride; a.kn_seq_stride = c.kn_seq_stride;
  a.v_seq_stride = c.v_seq_stride; a.vn_seq_stride = c.vn_seq_stride;
  a.k_head_stride = c.k_head_stride; a.kn_head_stride = c.kn_head_stride;
  a.v_head_stride = c.v_head_stride; a.vn_head_stride = c.vn_head_stride;
  a.split_len = plan.split_len;
  a.n_seq = c.n_seq; a.n_kv = c.n_kv_heads; a.n_rep = c.n_rep; a.n_splits = plan.n_splits; a.n_row_wgs = (int)row_wgs;
  a.causal = causal ? 1 : 0;
  a.q_dtype = c.q_dtype; a.out_dtype = c.out_dtype;
  a.q_wide = tq::aligned(c.q, 16); a.out_wide = tq::aligned(c.out, 16);
  Codebook kcb, vcb;
  const float k_unscale = tq::fill_codebook_fp16(kcb, c.k_centroids, c.bits);
  const float v_unscale = tq::fill_codebook_fp16(vcb, c.v_centroids, c.bits);
  a.score_scale = c.attn_scale / (float)c.dim * k_unscale * kLog2e;
  a.unscale = v_unscale / kVnScale / (float)c.dim;
  if (c.flags & TQ_PREFILL_FP16_QUERY) {
    TQ_DISPATCH_BITS(c.bits, (prefill_tile_kernel<B_, false><<<(unsigned)grid, kThreads, 0, c.stream>>>(a, kcb, vcb)));
  } else {
    TQ_DISPATCH_BITS(c.bits, (prefill_tile_kernel<B_><<<(unsigned)grid, kThreads, 0, c.stream>>>(a, kcb, vcb)));
  }
  TQ_CHECK_LAUNCH(who);
  if (plan.n_splits == 1) return TQ_OK;

  const int rgrid = (int)((rows + 4 * kRowsPerWavePass - 1) / (4 * kRowsPerWavePass));
  if (c.out_dtype == TQ_F32)
    prefill_merge_kernel<float><<<rgrid, 256, 0, c.stream>>>(a.ws_O, a.ws_ml, c.v_signs, (float*)c.out, (int64_t)rows,
                                                             plan.n_splits, a.unscale);
  else if (c.out_dtype == TQ_F16)
    prefill_merge_kernel<__half><<<rgrid, 256, 0, c.stream>>>(a.ws_O, a.ws_ml, c.v_signs, (__half*)c.out, (int64_t)rows,
                                                              plan.n_splits, a.unscale);
  else
    prefill_merge_kernel<__hip_bfloat16><<<rgrid, 256, 0, c.stream>>>(a.ws_O, a.ws_ml, c.v_signs, (__hip_bfloat16*)c.out,
                                                                      (int64_t)rows, plan.n_splits, a.unscale);
  TQ_CHECK_LAUNCH(who);
  return TQ_OK;
}

}  // namespace

// Splits of rows that all see the whole cache, a head of each kind a workgroup: what tq_prefill_attn has room for, which learns
// of the position of the chunk and of the heads that share keys only at the call (its plan may want more: the batch entry, whose
// size query knows them, gives it those).
static SplitPlan plan_any_position(int n_q_heads, int64_t n_rows, int64_t kv_len) {
  return plan_splits(1, n_q_heads, 1, n_rows, kv_len, 0, false, 32);
}

extern "C" size_t tq_prefill_workspace_bytes(int n_q_heads, int64_t n_rows, int64_t kv_len, int dim) {
  if (n_q_heads < 1 || n_rows < 1 || kv_len < 1 || dim != kD) return 0;
  return workspace_of(plan_any_position(n_q_heads, n_rows, kv_len).n_splits, (size_t)n_q_heads * (size_t)n_rows) + 512;
}

extern "C" size_t tq_prefill_batch_workspace_bytes(int n_seq, int n_kv_heads, int n_rep, int64_t n_rows, int64_t kv_len,
                                                   int64_t q_pos0, int dim, int flags) {
  if (n_seq < 1 || n_kv_heads < 1 || n_rep < 1 || n_rows < 1 || kv_len < 1 || q_pos0 < 0 || dim != kD) return 0;
  const bool causal = flags & TQ_PREFILL_CAUSAL;
  const SplitPlan p = plan_splits(n_seq, n_kv_heads, n_rep, n_rows, visible(kv_len, q_pos0, n_rows, causal), q_pos0, causal, 32);
  return workspace_of(p.n_splits, (size_t)n_seq * n_kv_heads * n_rep * (size_t)n_rows) + 512;
}

extern "C" int tq_prefill_attn(const void* q, int q_dtype, const uint32_t* k_packed, const float* k_norms,
                               const uint32_t* v_packed, const float* v_norms, const float* k_centroids,
                               const float* v_centroids, const float* k_signs, const float* v_signs, void* out,
                               int out_dtype, void* workspace, size_t workspace_bytes, int n_kv_heads, int n_rep,
                               int64_t n_rows, int64_t kv_len, int64_t q_pos0, int64_t k_head_stride,
                               int64_t kn_head_stride, int64_t v_head_stride, int64_t vn_head_stride, int dim,
                               int bits, float attn_scale, int flags, tq_stream_t stream) {
  const bool sizes = n_kv_heads > 0 && n_rep > 0 && n_rows > 0 && kv_len > 0;
  const size_t need = sizes ? tq_prefill_workspace_bytes(n_kv_heads * n_rep, n_rows, kv_len, dim) : 0;
  const int64_t most = sizes ? plan_any_position(n_kv_heads * n_rep, n_rows, kv_len).n_splits : 1;
  return prefill("tq_prefill_attn",
                 PrefillCall{q, q_dtype, k_packed, k_norms, v_packed, v_norms, k_centroids, v_centroids, k_signs, v_signs, out,
                             out_dtype, workspace, workspace_bytes, 1, n_kv_heads, n_rep, n_rows, kv_len, q_pos0, 0, 0, 0, 0,
                             k_head_stride, kn_head_stride, v_head_stride, vn_head_stride, dim, bits, attn_scale, flags,
                             (hipStream_t)stream},
                 need, most);
}

extern "C" int tq_prefill_attn_batch(const void* q, int q_dtype, const uint32_t* k_packed, const float* k_norms,
                                     const uint32_t* v_packed, const float* v_norms, const float* k_centroids,
                                     const float* v_centroids, const float* k_signs, const float* v_signs, void* out,
                                     int out_dtype, void* workspace, size_t workspace_bytes, int n_seq, int n_kv_heads,
                                     int n_rep, int64_t n_rows, int64_t kv_len, int64_t q_pos0, int64_t k_seq_stride,
                                     int64_t kn_seq_stride, int64_t v_seq_stride, int64_t vn_seq_stride,
                                     int64_t k_head_stride, int64_t kn_head_stride, int64_t v_head_stride,
                                     int64_t vn_head_stride, int dim, int bits, float attn_scale, int flags,
                                     tq_stream_t stream) {
  const size_t need = tq_prefill_batch_workspace_bytes(n_seq, n_kv_heads, n_rep, n_rows, kv_len, q_pos0, dim, flags);
  return prefill("tq_prefill_attn_batch",
                 PrefillCall{q, q_dtype, k_packed, k_norms, v_packed, v_norms, k_centroids, v_centroids, k_signs, v_signs, out,
                             out_dtype, workspace, workspace_bytes, n_seq, n_kv_heads, n_rep, n_rows, kv_len, q_pos0,
                             k_seq_stride, kn_seq_stride, v_seq_stride, vn_seq_stride, k_head_stride, kn_head_stride,
                             v_head_stride, vn_head_stride, dim, bits, attn_scale, flags, (hipStream_t)stream},
                 need, 32);
}
