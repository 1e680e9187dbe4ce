// Streaming encoder and dequantiser (d = 64, 128 and 256, 1 to 4 bits): d / 32 lanes own a vector, a wavefront works
// on 2048 elements (32, 16 or 8 vectors) per pass.  Included by the translation units that instantiate the kernels.
#pragma once

#include "tq_common.h"

namespace tqc {

using namespace tqd;

constexpr int kWavesPerBlock = 4;
constexpr int kBlock = kWavesPerBlock * TQ_WAVE;

struct Thresholds { float t[15]; };

// Rows of a call: n_rows = groups * rows_per_group; row r of group g of tensor X lies at g * X_group_stride + r.
// group_mul / group_shift: row / rows_per_group = mulhi(row, group_mul) >> group_shift for every row < 2^31
// (group_mul = 0: rows_per_group is 1).
struct RowMap {
  int64_t n_rows, rows_per_group, packed_group_stride, norms_group_stride, out_group_stride;
  uint32_t group_mul, group_shift;
};

// What an encode or dequantise launch reads and writes; a launch takes one such side, or the keys' and the values' of
// the same rows (blockIdx.y) with one RowMap, codebook and data type.
struct EncodeSide {
  const void* x;
  const float* signs;
  uint32_t* packed;
  float* norms;
};
struct DequantSide {
  const uint32_t* packed;
  const float* norms;
  const float* signs;
  void* out;
};
struct EncodeSides { EncodeSide s[2]; };
struct DequantSides { DequantSide s[2]; };

__device__ __forceinline__ void group_of(const RowMap& rm, uint32_t row, uint32_t& g, uint32_t& r) {
  g = rm.group_mul ? (__umulhi(row, rm.group_mul) >> rm.group_shift) : row;
  r = row - g * (uint32_t)rm.rows_per_group;
}

// alpha and beta of the level guess; beta0 = beta without the 2^20 + 32 that places the guess in the mantissa
struct EncodeGuess { float alpha, beta, beta0; };

// Mixed-precision FMA on one half of a packed fp16 pair (HI = 0: low half, 1: high half), so that fp16
// inputs need no separate widening instruction.  A product is taken as fma(a, b, -0): adding -0 changes
// no value, not even the sign of a zero, so it rounds exactly like the float32 multiply of the widened
// operands.
template <int HI>
__device__ __forceinline__ float mix_sq(uint32_t h2, float negzero) {           // widen(h) * widen(h)
  float d;
  if (HI) asm("v_fma_mix_f32 %0, %1, %1, %2 op_sel:[1,1,0] op_sel_hi:[1,1,0]" : "=v"(d) : "v"(h2), "v"(negzero));
  else    asm("v_fma_mix_f32 %0, %1, %1, %2 op_sel:[0,0,0] op_sel_hi:[1,1,0]" : "=v"(d) : "v"(h2), "v"(negzero));
  return d;
}
template <int HI>
__device__ __forceinline__ float mix_mul(uint32_t h2, float b, float negzero) { // widen(h) * b
  float d;
  if (HI) asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d) : "v"(h2), "v"(b), "v"(negzero));
  else    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(d) : "v"(h2), "v"(b), "v"(negzero));
  return d;
}
template <int HI>
__device__ __forceinline__ float mix_fma_addend(float a, float b, uint32_t h2) { // fma(a, b, widen(h))
  float d;
  if (HI) asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(d) : "v"(a), "v"(b), "v"(h2));
  else    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,0] op_sel_hi:[0,0,1]" : "=v"(d) : "v"(a), "v"(b), "v"(h2));
  return d;
}

// The 8 * BITS bits that hold elements 8c .. 8c+7 (chunk c) of a packed row of D fields: word and shifts.  Three-bit
// rows hold ten fields per word, so a chunk may straddle two words (chunk 15 of a d = 128 row is all of word 12:
// taken as word 11 >> 30, which is 0, | word 12); the other widths divide the word.
template <int D, int BITS>
struct Chunk {
  static constexpr int kPd = Pk<BITS>::pdim(D);                // words per row
  static constexpr uint32_t kPairMask = (1u << (2 * BITS)) - 1u;
  __device__ static __forceinline__ void pos(int c, int& w0, int& sh_lo, int& sh_hi) {
    if (BITS == 3) {
      const bool last = D == 128 && c == 15;
      w0 = last ? 11 : (8 * c) / 10;
      const int s0 = last ? 10 : (8 * c) % 10;
      sh_lo = 3 * s0;
      sh_hi = 30 - 3 * s0;
    } else {
      constexpr int kPerWord = 4 / BITS;
      w0 = c / kPerWord;
      sh_lo = (c % kPerWord) * 8 * BITS;
      sh_hi = 0;
    }
  }
  __device__ static __forceinline__ uint32_t field(const uint32_t* at_w0, int sh_lo, int sh_hi) {
    if constexpr (BITS == 3) return ((at_w0[0] >> sh_lo) | (at_w0[1] << sh_hi)) & 0xFFFFFFu;
    else if constexpr (BITS == 4) return at_w0[0];
    else return (at_w0[0] >> sh_lo) & ((1u << (8 * BITS)) - 1u);
  }
};

constexpr int kEncPasses = 4;     // passes per wavefront once there are rows enough to fill the chip

// Encoder.  Lane ls of a vector holds its four 8-element chunks c = ls + kLanes k (k = 0..3), element
// e = 8 kLanes k + 8 ls + j (VecLanes).  Each load instruction therefore reads 16 kLanes contiguous bytes per vector;
// butterfly stages 1, 2, 4 and the two largest, and the first two and last three levels of the sum-of-squares tree
// stay inside a lane, and the stages between are lane exchanges folded into the add.  Results are bit-identical to
// encode_kernel:
//  * the sum of squares is added in the same stride-halving tree order;
//  * x / n is computed as q = x*r, q += r * fma(-n, q, x) with r = 1/n correctly rounded, which
//    yields the correctly rounded quotient (checked against IEEE division on 3e10 operand pairs
//    with |x| <= n), at 3 operations per element instead of a full division;
//  * the count of thresholds exceeded is g + (w > t[g]) where g is a guess that the host has verified to be
//    the count or one less for every w: v = fma(w, alpha, beta + 2^20 + 32) lies in [2^20, 2^21), where
//    floats are 1/8 apart, so bits 3..8 of v are 32 + floor(alpha*w + beta) (to within the rounding to
//    1/8) and, masked, are the byte offset into a 64-entry LDS table of (t[g], g) pairs whose entries
//    below / above the seven levels hold (+inf, 0) / (-inf, 6): no clamp (at d = 256, where |w| may reach 16, one
//    median instruction), no float-to-int convert, no address shift.  A NaN norm forces all indices of the vector
//    to 0 (as comparisons with NaN do).
// Packed words leave through LDS so that a wavefront stores up to 256 contiguous words per pass.
//
// BITS = 3: every threshold j sits in cell j of the guess (level_guess_search), and the table is written down
// directly.  Other widths: any guess line under which no cell holds two thresholds (level_cells_search); cell
// c = floor(alpha * w + beta0) then knows the count g of thresholds below its lower edge and the one threshold it
// may hold (else +inf: nothing to compare with), both derived here from the thresholds themselves.
//
// RAGGED = false: rows_per_group is a multiple of the vectors of a pass, so a pass lies inside one group and its
// destination rows are consecutive.  RAGGED = true takes any row count (a prompt's length is no multiple of
// anything): a pass takes the next kVecs rows whatever their groups, every lane derives its own vector's group once
// per pass and the destination rows of the pass are shared through LDS; rows past the end repeat the last one and
// are not stored.  What it costs over the other form is a dozen instructions per 2048 elements.
//
// INDICES: the levels leave as one byte each instead of packed words, `packed` standing for n_rows x D bytes without groups
// (RAGGED).  Bound as the packing form is (256 bytes in, 132 out per fp16 row of 128): 100 003 rows in one launch 12.4 - 13.6 us by the box,
// against 12.7 us of encoding and 5.4 us of unpacking the words again.
template <int D, typename T, int BITS, bool RAGGED, bool INDICES = false>
__global__ __launch_bounds__(kBlock) void encode_rows_kernel(EncodeSides sides, Thresholds thr, EncodeGuess gs, RowMap rm,
                                                             int passes) {
  const T* __restrict__ x = (const T*)sides.s[blockIdx.y].x;
  const float* __restrict__ signs = sides.s[blockIdx.y].signs;
  uint32_t* __restrict__ packed = sides.s[blockIdx.y].packed;
  float* __restrict__ norms = sides.s[blockIdx.y].norms;
  using VL = VecLanes<D>;
  constexpr int kLanes = VL::kLanes, kVecs = VL::kVecs, kChunks = D / 8;
  constexpr bool kHalfWidth = sizeof(T) == 2;
  constexpr int NM = kHalfWidth ? 4 : 8;                       // sign masks per chunk
  constexpr int NB = (1 << BITS) - 1;                          // thresholds
  constexpr int kPd = Chunk<D, BITS>::kPd;
  constexpr int kCells = BITS == 4 ? 128 : 64;                 // cells of the level guess (fifteen thresholds need finer ones)
  __shared__ __align__(8) uint2 lvl_s[kCells];                 // (threshold bits, guess) by kCells / 2 + floor(alpha*w + beta0)
  __shared__ __align__(16) float sg_s[D];
  constexpr int kIdxPitch = D + 16;                            // bytes per row of indices in LDS: conflict-free 8-byte writes
  __shared__ __align__(16) uint32_t chunk_s[kWavesPerBlock][INDICES ? kVecs * kIdxPitch / 4 : kVecs * kChunks + 4];
  __shared__ uint32_t dst_s[kWavesPerBlock][RAGGED && !INDICES ? kVecs : 1];   // destination row of each vector of the pass

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ls = VL::logical(lane), v = lane / kLanes;
  if (tid < kCells) {
    const int gq = tid - kCells / 2;
    if (BITS == 3) {
      float t = gq < 0 ? INFINITY : -INFINITY;
#pragma unroll
      for (int i = 0; i < 7; ++i) t = (gq == i) ? thr.t[i] : t;
      lvl_s[tid] = make_uint2(__float_as_uint(t), (uint32_t)(gq < 0 ? 0 : (gq > 6 ? 6 : gq)));
    } else {
      int g = 0;                                               // thresholds below the cell's lower edge
#pragma unroll
      for (int i = 0; i < NB; ++i) g += (__fmaf_rn(thr.t[i], gs.alpha, gs.beta0) < (float)gq) ? 1 : 0;
      float t = INFINITY;                                      // threshold number g, if it lies inside the cell
#pragma unroll
      for (int i = 0; i < NB; ++i)
        t = (i == g && __fmaf_rn(thr.t[i], gs.alpha, gs.beta0) < (float)(gq + 1)) ? thr.t[i] : t;
      lvl_s[tid] = make_uint2(__float_as_uint(t), (uint32_t)g);
    }
  }
  if (tid < D) sg_s[tid] = signs[tid];
  __syncthreads();

  // sign flips as xor masks on the raw input bits
  uint32_t sm[4][NM];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float4 a = *reinterpret_cast<const float4*>(&sg_s[8 * kLanes * k + 8 * ls]);
    const float4 b = *reinterpret_cast<const float4*>(&sg_s[8 * kLanes * k + 8 * ls + 4]);
    const float sv[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    if (kHalfWidth) {
#pragma unroll
      for (int jp = 0; jp < 4; ++jp)
        sm[k][jp] = ((__float_as_uint(sv[2 * jp]) >> 16) & 0x8000u) | (__float_as_uint(sv[2 * jp + 1]) & 0x80000000u);
    } else {
#pragma unroll
      for (int j = 0; j < NM; ++j) sm[k][j] = __float_as_uint(sv[j & 7]) & 0x80000000u;
    }
  }
  // lanes with an odd number of bits in ls take their inputs negated (folded into the sign masks): butterfly_lanes_neg
  if (__popc(ls) & 1) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int j = 0; j < NM; ++j) sm[k][j] ^= kHalfWidth ? 0x80008000u : 0x80000000u;
  }
  const float m[3] = {(ls & 1) ? 1.0f : -1.0f, (ls & 2) ? 1.0f : -1.0f, (ls & 4) ? 1.0f : -1.0f};
  uint32_t* chunks = chunk_s[wave];

  // first batch of kVecs rows of this wavefront and, where a batch lies inside one group, its place in the (group, row) map
  const uint32_t n_rows = (uint32_t)rm.n_rows;
  const uint32_t batch0 = ((uint32_t)blockIdx.x * kWavesPerBlock + wave) * (uint32_t)passes;
  uint32_t row0 = batch0 * kVecs;
  uint32_t grp = 0, rin = 0;
  if (!RAGGED) {
    grp = row0 / (uint32_t)rm.rows_per_group;
    rin = row0 - grp * (uint32_t)rm.rows_per_group;
  }
  auto row_ptr = [&](uint32_t first) {                         // this lane's first chunk of its vector of the pass at `first`
    uint32_t row = first + v;
    if (RAGGED) row = min(row, n_rows - 1);
    return x + (int64_t)row * D + 8 * ls;
  };

  // 16-bit inputs: the rows of the next pass are fetched while the current one is computed
  uint4 nraw[4] = {};
  if (kHalfWidth && row0 < n_rows) {
    const T* xr = row_ptr(row0);
#pragma unroll
    for (int k = 0; k < 4; ++k) nraw[k] = *reinterpret_cast<const uint4*>(xr + 8 * kLanes * k);
  }
  for (int pass = 0; pass < passes; ++pass) {
    if (row0 >= n_rows) break;                                 // uniform over the wavefront
    // ---- load, flip signs, widen (fp16: the packed pairs stay as they are and are widened inside the
    // mixed-precision multiplies below)
    constexpr bool kMix = __is_same(T, __half);
    float xs[4][8];
    uint32_t hw[4][4];
    if (kHalfWidth) {
      uint4 raw[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) raw[k] = nraw[k];
      if (pass + 1 < passes && row0 + kVecs < n_rows) {
        const T* xr = row_ptr(row0 + kVecs);
#pragma unroll
        for (int k = 0; k < 4; ++k) nraw[k] = *reinterpret_cast<const uint4*>(xr + 8 * kLanes * k);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t w[4] = {raw[k].x ^ sm[k][0], raw[k].y ^ sm[k][1], raw[k].z ^ sm[k][2], raw[k].w ^ sm[k][3]};
#pragma unroll
        for (int jp = 0; jp < 4; ++jp) {
          hw[k][jp] = w[jp];
          if (!kMix) {
            xs[k][2 * jp] = __uint_as_float(w[jp] << 16);
            xs[k][2 * jp + 1] = __uint_as_float(w[jp] & 0xFFFF0000u);
          }
        }
      }
    } else {
      const T* xr = row_ptr(row0);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint4 a = *reinterpret_cast<const uint4*>(xr + 8 * kLanes * k);
        const uint4 b = *reinterpret_cast<const uint4*>(xr + 8 * kLanes * k + 4);
        const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int j = 0; j < 8; ++j) xs[k][j] = __uint_as_float(w[j] ^ sm[k][j & (NM - 1)]);
      }
    }
    // ---- where this lane's vector goes
    uint32_t my_g = grp, my_r = rin + v;
    const bool mine = !RAGGED || row0 + v < n_rows;
    if (INDICES) {
      my_g = 0;
      my_r = row0 + v;
    } else if (RAGGED) {
      group_of(rm, min(row0 + v, n_rows - 1), my_g, my_r);
      dst_s[wave][v] = my_g * (uint32_t)rm.packed_group_stride + my_r;
    }
    const float negzero = -0.0f;
    // ---- sum of squares: the two largest strides (k), the lanes, then 4, 2, 1 (j)
    float t8[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float sq[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (kMix) sq[k] = (j & 1) ? mix_sq<1>(hw[k][j >> 1], negzero) : mix_sq<0>(hw[k][j >> 1], negzero);
        else sq[k] = xs[k][j] * xs[k][j];
      }
      t8[j] = (sq[0] + sq[2]) + (sq[1] + sq[3]);
    }
    if constexpr (kLanes >= 8) {
#pragma unroll
      for (int j = 0; j < 8; ++j) t8[j] = t8[j] + oct_mirror(t8[j]);
    }
    if constexpr (kLanes >= 4) {
#pragma unroll
      for (int j = 0; j < 8; ++j) t8[j] = t8[j] + quad_xor2(t8[j]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) t8[j] = t8[j] + quad_xor1(t8[j]);
    const float ss = ((t8[0] + t8[4]) + (t8[2] + t8[6])) + ((t8[1] + t8[5]) + (t8[3] + t8[7]));
    const float nrm = sqrtf(ss);
    const float safe = fmaxf(nrm, 1e-8f);
    const float rinv = 1.0f / safe;
    // a norm that overflowed to infinity: x / inf is 0 for every finite x, which q = x * 0 already is; the
    // correction term must then not multiply infinity by that zero
    const float nsafe = (safe == INFINITY) ? 0.0f : -safe;
    // ---- unit vector
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (kMix) {
          const uint32_t h2 = hw[k][j >> 1];
          const float q0 = (j & 1) ? mix_mul<1>(h2, rinv, negzero) : mix_mul<0>(h2, rinv, negzero);
          const float rem = (j & 1) ? mix_fma_addend<1>(nsafe, q0, h2) : mix_fma_addend<0>(nsafe, q0, h2);
          xs[k][j] = __fmaf_rn(rem, rinv, q0);
        } else {
          const float q0 = xs[k][j] * rinv;
          const float rem = __fmaf_rn(nsafe, q0, xs[k][j]);
          xs[k][j] = __fmaf_rn(rem, rinv, q0);
        }
      }
    butterfly_lanes_neg<kLanes>(xs, m);
    // ---- levels, 8 * BITS bits per chunk
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      uint32_t bits24 = 0, top4 = 0;                           // INDICES: bytes of elements 0 .. 3 and 4 .. 7
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float w = xs[k][j];
        float cell = __fmaf_rn(w, gs.alpha, gs.beta);
        if (D > 128)                                           // |w| <= 16 may leave the table: into its first or last cell
          cell = __builtin_amdgcn_fmed3f(cell, 1048576.0f, 1048576.0f + (float)(kCells - 1));
        const uint32_t off = __float_as_uint(cell) & (uint32_t)((kCells - 1) << 3);
        const uint2 lv = *reinterpret_cast<const uint2*>(reinterpret_cast<const unsigned char*>(lvl_s) + off);
        const uint32_t idx = lv.y + ((w > __uint_as_float(lv.x)) ? 1u : 0u);
        if constexpr (INDICES) (j < 4 ? bits24 : top4) |= idx << (8 * (j & 3));
        else bits24 |= idx << (BITS * j);
      }
      if constexpr (INDICES)
        *reinterpret_cast<uint2*>(reinterpret_cast<unsigned char*>(chunks) + v * kIdxPitch + 8 * (ls + kLanes * k)) =
            (nrm != nrm) ? make_uint2(0u, 0u) : make_uint2(bits24, top4);
      else
        chunks[v * kChunks + ls + kLanes * k] = (nrm != nrm) ? 0u : bits24;
    }
    wave_lds_fence();
    if constexpr (INDICES) {                                   // 1 KB of consecutive bytes per store instruction
      unsigned char* rows = reinterpret_cast<unsigned char*>(packed) + (int64_t)row0 * D;
#pragma unroll
      for (int it = 0; it < 2; ++it) {
        const int piece = it * 64 + lane, vv = piece / (D / 16);
        const uint4 val = *reinterpret_cast<const uint4*>(reinterpret_cast<const unsigned char*>(chunks) + vv * kIdxPitch + 16 * (piece % (D / 16)));
        if (row0 + vv < n_rows) *reinterpret_cast<uint4*>(rows + 16 * piece) = val;
      }
      wave_lds_fence();
      if (ls == 0 && mine) norms[my_r] = nrm;
      row0 += kVecs;
      continue;
    }
    // ---- words.  Three bits: word wd of a row holds elements 10wd .. 10wd+9 = chunks (5wd)/4 and the next;
    // four bits: a chunk is a word; two bits / one bit: two / four chunks make a word
    uint32_t* prow = packed + ((int64_t)grp * rm.packed_group_stride + rin) * kPd;
#pragma unroll
    for (int it = 0; it < (kVecs * kPd + 63) / 64; ++it) {
      const int id = it * 64 + lane;
      if (id < kVecs * kPd) {
        const int vv = id / kPd, wd = id - kPd * vv;
        uint32_t word;
        if constexpr (BITS == 3) {
          constexpr uint32_t kLastMask = (1u << (3 * (D - 10 * (kPd - 1)))) - 1u;   // the last word holds what is left of D
          const int a = (5 * wd) >> 2, sh = 3 * ((10 * wd) & 7);
          const uint32_t lo = chunks[vv * kChunks + a], hi = chunks[vv * kChunks + a + 1];
          word = ((lo >> sh) | (hi << (24 - sh))) & (wd == kPd - 1 ? kLastMask : 0x3FFFFFFFu);
        } else if constexpr (BITS == 4) {
          word = chunks[vv * kChunks + wd];
        } else if constexpr (BITS == 2) {
          word = chunks[vv * kChunks + 2 * wd] | (chunks[vv * kChunks + 2 * wd + 1] << 16);
        } else {
          word = chunks[vv * kChunks + 4 * wd] | (chunks[vv * kChunks + 4 * wd + 1] << 8) |
                 (chunks[vv * kChunks + 4 * wd + 2] << 16) | (chunks[vv * kChunks + 4 * wd + 3] << 24);
        }
        if (!RAGGED) prow[id] = word;
        else if (row0 + vv < n_rows) packed[(int64_t)dst_s[wave][vv] * kPd + wd] = word;
      }
    }
    wave_lds_fence();                                          // the next pass overwrites chunks and destinations
    if (ls == 0 && mine) norms[(int64_t)my_g * rm.norms_group_stride + my_r] = nrm;
    row0 += kVecs;
    if (!RAGGED) {
      rin += kVecs;
      if (rin >= (uint32_t)rm.rows_per_group) { rin = 0; ++grp; }
    }
  }
}

// Dequantiser: the same lanes per vector, every width.  The packed words of a pass (208 at d = 128 and three bits) are
// read with coalesced loads into LDS; a lane cuts the 8 * BITS bits of each of its chunks out of one or two words and
// looks centroid pairs up in a table of 4^BITS entries (c[a]*s, c[b]*s).  Arithmetic per element, in this order, as in
// dequant_kernel: butterfly, * s, * sign, * norm, round to TO.  RAGGED as in the encoder.
//
// INDICES: the levels come as one byte each, `packed` standing for n_rows x D bytes without groups (RAGGED).  A lane reads its
// chunks as they lie (8 bytes each, 16 kLanes bytes of a row per instruction) and looks pairs up from them.  Bytes past the width
// mean what packing them first would give: words of the summed, shifted bytes, cut to `word_bits` (three bits: whether the two
// bits above a word's ten fields reach the next chunk depends on the kernel that reads the words); a wavefront that meets one
// builds the words of its pass.  100 003 rows of 128 to float32 13.2 - 13.6 us against 8.1 us of packing and 11.6 us of this kernel
// on the words.
template <int D, typename TO, int BITS, bool RAGGED, bool INDICES = false>
__global__ __launch_bounds__(kBlock) void dequant_rows_kernel(DequantSides sides, Codebook cbk, float s, RowMap rm,
                                                              int passes, uint32_t word_bits = ~0u) {
  const uint32_t* __restrict__ packed = sides.s[blockIdx.y].packed;
  const float* __restrict__ norms = sides.s[blockIdx.y].norms;
  const float* __restrict__ signs = sides.s[blockIdx.y].signs;
  TO* __restrict__ out = (TO*)sides.s[blockIdx.y].out;
  using CK = Chunk<D, BITS>;
  using VL = VecLanes<D>;
  constexpr int kLanes = VL::kLanes, kVecs = VL::kVecs;
  constexpr int kPd = CK::kPd;
  constexpr int kPairs = 1 << (2 * BITS);                      // entries of the centroid-pair table
  constexpr int kWordLoads = (kVecs * kPd + 63) / 64;          // wave-wide loads of a pass's packed words
  __shared__ __align__(16) float sg_s[D];
  // centroid pairs, and after them the same pairs negated: lanes with an odd number of bits in ls read those
  // (butterfly_lanes_neg)
  __shared__ __align__(8) float2 pair_s[2 * kPairs];
  __shared__ uint32_t words_s[kWavesPerBlock][kVecs * kPd + 3];
  constexpr bool kMapped = RAGGED && !INDICES;
  __shared__ uint32_t src_s[kWavesPerBlock][kMapped ? kVecs : 1], dst_s[kWavesPerBlock][kMapped ? kVecs : 1];
  // Outputs leave through LDS: rows at a padded pitch (conflict-free 16-byte writes per lane and reads per row
  // segment), so that every store instruction writes 1 KB of contiguous memory
  constexpr int kPiecesPerRow = D * (int)sizeof(TO) / 16;
  constexpr int kPitch = 16 * (sizeof(TO) == 2 ? kPiecesPerRow + kLanes : kPiecesPerRow + 1);
  __shared__ __align__(16) unsigned char orow_s[kWavesPerBlock][kVecs * kPitch];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ls = VL::logical(lane), v = lane / kLanes;
  if (tid < kPairs) {                                          // kBlock = 256 threads cover the largest table
    float clo = 0.0f, chi = 0.0f;
#pragma unroll
    for (int i = 0; i < (1 << BITS); ++i) {
      clo = ((tid & ((1 << BITS) - 1)) == i) ? cbk.c[i] : clo;
      chi = ((tid >> BITS) == i) ? cbk.c[i] : chi;
    }
    pair_s[tid] = make_float2(clo * s, chi * s);
    pair_s[kPairs + tid] = make_float2(-(clo * s), -(chi * s));
  }
  if (tid >= kBlock - D) sg_s[tid - (kBlock - D)] = signs[tid - (kBlock - D)];
  __syncthreads();

  uint32_t sm[4][8];                                           // sign bit of each element of this lane
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float4 a = *reinterpret_cast<const float4*>(&sg_s[8 * kLanes * k + 8 * ls]);
    const float4 b = *reinterpret_cast<const float4*>(&sg_s[8 * kLanes * k + 8 * ls + 4]);
    const float sv[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) sm[k][j] = __float_as_uint(sv[j]) & 0x80000000u;
  }
  const float m[3] = {(ls & 1) ? 1.0f : -1.0f, (ls & 2) ? 1.0f : -1.0f, (ls & 4) ? 1.0f : -1.0f};
  const float2* my_pairs = pair_s + ((__popc(ls) & 1) ? kPairs : 0);
  uint32_t* words = words_s[wave];
  // words / shifts of the bits of chunk c = ls + kLanes k (elements 8c .. 8c+7)
  int cw[4], csl[4], csh[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) CK::pos(ls + kLanes * k, cw[k], csl[k], csh[k]);

  const uint32_t n_rows = (uint32_t)rm.n_rows;
  const uint32_t batch0 = ((uint32_t)blockIdx.x * kWavesPerBlock + wave) * (uint32_t)passes;
  uint32_t row0 = batch0 * kVecs;
  uint32_t grp = 0, rin = 0;
  if (!RAGGED) {
    grp = row0 / (uint32_t)rm.rows_per_group;
    rin = row0 - grp * (uint32_t)rm.rows_per_group;
  }

  // the packed words and the norm of the next pass are fetched while the current one is computed
  uint32_t pw[kWordLoads];
  float pn = 0.0f;
  uint32_t my_out = 0;                                         // RAGGED: output row of this lane's vector in the fetched pass
  uint2 pi[4];                                                 // INDICES: bytes of this lane's chunks
  const uint8_t* ibytes = reinterpret_cast<const uint8_t*>(packed);
  auto fetch = [&](uint32_t first, uint32_t g_, uint32_t r_) {
    if constexpr (INDICES) {
      const uint32_t row = min(first + v, n_rows - 1);
      pn = norms[row];
      const uint8_t* src = ibytes + (int64_t)row * D + 8 * ls;
#pragma unroll
      for (int k = 0; k < 4; ++k) pi[k] = *reinterpret_cast<const uint2*>(src + 8 * kLanes * k);
    } else if (RAGGED) {
      uint32_t mg, mr;
      group_of(rm, min(first + v, n_rows - 1), mg, mr);
      src_s[wave][v] = mg * (uint32_t)rm.packed_group_stride + mr;
      wave_lds_fence();
      my_out = mg * (uint32_t)rm.out_group_stride + mr;
      pn = norms[(int64_t)mg * rm.norms_group_stride + mr];
#pragma unroll
      for (int it = 0; it < kWordLoads; ++it) {
        const int id = it * 64 + lane;
        const int vv = min(id / kPd, kVecs - 1), wd = min(id - kPd * vv, kPd - 1);
        pw[it] = packed[(int64_t)src_s[wave][vv] * kPd + wd];
      }
    } else {
      const uint32_t* prow = packed + ((int64_t)g_ * rm.packed_group_stride + r_) * kPd;
      pn = norms[(int64_t)g_ * rm.norms_group_stride + r_ + v];
#pragma unroll
      for (int it = 0; it < kWordLoads; ++it) {
        const int id = it * 64 + lane;
        pw[it] = (id < kVecs * kPd) ? prow[id] : 0u;
      }
    }
  };
  if (row0 < n_rows) fetch(row0, grp, rin);
  for (int pass = 0; pass < passes; ++pass) {
    if (row0 >= n_rows) break;                                 // uniform over the wavefront
    const float nrm = pn;
    uint2 ib[4];
    if constexpr (INDICES) {
#pragma unroll
      for (int k = 0; k < 4; ++k) ib[k] = pi[k];
    } else {
      if (RAGGED) dst_s[wave][v] = my_out;
#pragma unroll
      for (int it = 0; it < kWordLoads; ++it) {
        const int id = it * 64 + lane;
        if (id < kVecs * kPd) words[id] = pw[it];
      }
    }
    uint32_t nrin = rin + kVecs, ngrp = grp;
    if (!RAGGED && nrin >= (uint32_t)rm.rows_per_group) { nrin = 0; ++ngrp; }
    if (!INDICES) wave_lds_fence();
    if (pass + 1 < passes && row0 + kVecs < n_rows) fetch(row0 + kVecs, ngrp, nrin);
    float xs[4][8];
    bool from_words = !INDICES;
    if constexpr (INDICES) {
      uint32_t past = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) past |= ib[k].x | ib[k].y;
      from_words = __any((past & (0x01010101u * (0x100u - (1u << BITS)))) != 0);
      if (from_words) {
        constexpr int VPW = Pk<BITS>::VPW;
        for (int id = lane; id < kVecs * kPd; id += 64) {
          const int vv = id / kPd, e0 = (id - vv * kPd) * VPW;
          const uint8_t* src = ibytes + (int64_t)min(row0 + vv, n_rows - 1) * D + e0;
          uint32_t word = 0;
          for (int i = 0; i < min(VPW, D - e0); ++i) word += (uint32_t)src[i] << (BITS * i);
          words[id] = word & word_bits;
        }
        wave_lds_fence();
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int jp = 0; jp < 4; ++jp) {
            const uint32_t b4 = jp < 2 ? ib[k].x : ib[k].y;
            const float2 c2 = my_pairs[((b4 | (b4 >> (8 - BITS))) >> (16 * (jp & 1))) & CK::kPairMask];
            xs[k][2 * jp] = c2.x;
            xs[k][2 * jp + 1] = c2.y;
          }
      }
    }
    if (from_words) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t f = CK::field(words + v * kPd + cw[k], csl[k], csh[k]);
#pragma unroll
        for (int jp = 0; jp < 4; ++jp) {
          const float2 c2 = my_pairs[(f >> (2 * BITS * jp)) & CK::kPairMask];
          xs[k][2 * jp] = c2.x;
          xs[k][2 * jp + 1] = c2.y;
        }
      }
    }
    butterfly_lanes_neg<kLanes>(xs, m);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float r[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float t = (xs[k][j] * s) * nrm;
        asm volatile("" : "+v"(t));                            // keep the multiply out of the narrowing convert
        r[j] = t;
      }
      if (sizeof(TO) == 4) {
        uint4 a, b;
        a.x = __float_as_uint(r[0]) ^ sm[k][0]; a.y = __float_as_uint(r[1]) ^ sm[k][1];
        a.z = __float_as_uint(r[2]) ^ sm[k][2]; a.w = __float_as_uint(r[3]) ^ sm[k][3];
        b.x = __float_as_uint(r[4]) ^ sm[k][4]; b.y = __float_as_uint(r[5]) ^ sm[k][5];
        b.z = __float_as_uint(r[6]) ^ sm[k][6]; b.w = __float_as_uint(r[7]) ^ sm[k][7];
        *reinterpret_cast<uint4*>(&orow_s[wave][v * kPitch + 32 * kLanes * k + 32 * ls]) = a;
        *reinterpret_cast<uint4*>(&orow_s[wave][v * kPitch + 32 * kLanes * k + 32 * ls + 16]) = b;
      } else {
        uint32_t w[4];
#pragma unroll
        for (int jp = 0; jp < 4; ++jp) {
          uint32_t lo, hi;
          if (__is_same(TO, __half)) {
            lo = __half_as_ushort(__float2half_rn(r[2 * jp]));
            hi = __half_as_ushort(__float2half_rn(r[2 * jp + 1]));
          } else {
            lo = __bfloat16_as_ushort(__float2bfloat16(r[2 * jp]));
            hi = __bfloat16_as_ushort(__float2bfloat16(r[2 * jp + 1]));
          }
          w[jp] = (lo | (hi << 16)) ^ ((sm[k][2 * jp] >> 16) | sm[k][2 * jp + 1]);
        }
        *reinterpret_cast<uint4*>(&orow_s[wave][v * kPitch + 16 * kLanes * k + 16 * ls]) = make_uint4(w[0], w[1], w[2], w[3]);
      }
    }
    wave_lds_fence();
    {
      // streaming stores (the "nt" hint): the rows are not read again by this kernel and a pass writes more than the
      // caches hold -- 115 -> 99 us per 1 M float32 rows, 75 -> 66 us for fp16 (d = 128)
      typedef uint32_t piece_t __attribute__((ext_vector_type(4)));
      unsigned char* oblock = reinterpret_cast<unsigned char*>(
          out + (INDICES ? (int64_t)row0 * D : RAGGED ? 0 : ((int64_t)grp * rm.out_group_stride + rin) * D));
#pragma unroll
      for (int i = 0; i < (int)(2 * sizeof(TO)); ++i) {            // 4 or 8 KB per pass
        const int piece = i * 64 + lane;
        const int vv = piece / kPiecesPerRow, pc = piece % kPiecesPerRow;
        const piece_t val = *reinterpret_cast<const piece_t*>(&orow_s[wave][vv * kPitch + pc * 16]);
        if (!kMapped) {
          if (!RAGGED || row0 + vv < n_rows) __builtin_nontemporal_store(val, reinterpret_cast<piece_t*>(oblock + piece * 16));
        } else if (row0 + vv < n_rows) {
          __builtin_nontemporal_store(val, reinterpret_cast<piece_t*>(oblock + ((int64_t)dst_s[wave][vv] * kPiecesPerRow + pc) * 16));
        }
      }
    }
    wave_lds_fence();
    row0 += kVecs;
    rin = nrin;
    grp = ngrp;
  }
}

// ---------------------------------------------------------------- launches

struct EncodeCall {
  EncodeSides sides;
  int n_sides;
  int x_dtype;
  Thresholds thr;
  EncodeGuess gs;
  RowMap rm;
  int bits;
  hipStream_t stream;
};
struct DequantCall {
  DequantSides sides;
  int n_sides;
  Codebook cb;
  float s;
  int out_dtype;
  RowMap rm;
  int bits;
  hipStream_t stream;
};

// Passes per wavefront: several, to spread the set-up cost, once every CU has a few workgroups anyway.
template <int D>
inline int stream_passes(int64_t n_rows) {
  const int64_t rows_per_block_pass = (int64_t)VecLanes<D>::kVecs * kWavesPerBlock;
  return (n_rows >= rows_per_block_pass * kEncPasses * 256 * 4) ? kEncPasses : 1;
}
template <int D>
inline int stream_grid(int64_t n_rows, int passes) {
  const int64_t rows_per_block = (int64_t)VecLanes<D>::kVecs * passes * kWavesPerBlock;
  return (int)((n_rows + rows_per_block - 1) / rows_per_block);
}

template <int D, bool RAGGED>
void launch_encode_rows(const EncodeCall& c) {
  const int passes = stream_passes<D>(c.rm.n_rows * c.n_sides);
  const dim3 grid(stream_grid<D>(c.rm.n_rows, passes), c.n_sides);
#define TQ_LAUNCH_ENC(T)                                                                                             \
  TQ_DISPATCH_BITS(c.bits, (encode_rows_kernel<D, T, B_, RAGGED><<<grid, kBlock, 0, c.stream>>>(                      \
                               c.sides, c.thr, c.gs, c.rm, passes)))
  if (c.x_dtype == TQ_F32) { TQ_LAUNCH_ENC(float); }
  else if (c.x_dtype == TQ_F16) { TQ_LAUNCH_ENC(__half); }
  else { TQ_LAUNCH_ENC(__hip_bfloat16); }
#undef TQ_LAUNCH_ENC
}

template <int D, bool RAGGED>
void launch_dequant_rows(const DequantCall& c) {
  const int passes = stream_passes<D>(c.rm.n_rows * c.n_sides);
  const dim3 grid(stream_grid<D>(c.rm.n_rows, passes), c.n_sides);
#define TQ_LAUNCH_DEQ(TO)                                                                                            \
  TQ_DISPATCH_BITS(c.bits, (dequant_rows_kernel<D, TO, B_, RAGGED><<<grid, kBlock, 0, c.stream>>>(                    \
                               c.sides, c.cb, c.s, c.rm, passes)))
  if (c.out_dtype == TQ_F32) { TQ_LAUNCH_DEQ(float); }
  else if (c.out_dtype == TQ_F16) { TQ_LAUNCH_DEQ(__half); }
  else { TQ_LAUNCH_DEQ(__hip_bfloat16); }
#undef TQ_LAUNCH_DEQ
}

// levels as bytes: any number of rows, no groups
template <int D>
void launch_encode_indices(const EncodeCall& c) {
  const int passes = stream_passes<D>(c.rm.n_rows);
  const int grid = stream_grid<D>(c.rm.n_rows, passes);
#define TQ_LAUNCH_ENC(T)                                                                                             \
  TQ_DISPATCH_BITS(c.bits, (encode_rows_kernel<D, T, B_, true, true><<<grid, kBlock, 0, c.stream>>>(                  \
                               c.sides, c.thr, c.gs, c.rm, passes)))
  if (c.x_dtype == TQ_F32) { TQ_LAUNCH_ENC(float); }
  else if (c.x_dtype == TQ_F16) { TQ_LAUNCH_ENC(__half); }
  else { TQ_LAUNCH_ENC(__hip_bfloat16); }
#undef TQ_LAUNCH_ENC
}
template <int D>
void launch_dequant_indices(const DequantCall& c, uint32_t word_bits) {
  const int passes = stream_passes<D>(c.rm.n_rows);
  const int grid = stream_grid<D>(c.rm.n_rows, passes);
  TQ_DISPATCH_BITS(c.bits, (dequant_rows_kernel<D, float, B_, true, true><<<grid, kBlock, 0, c.stream>>>(
                               c.sides, c.cb, c.s, c.rm, passes, word_bits)));
}

// instantiated in translation units of their own, in parallel with the rest of the build
extern template void launch_encode_rows<64, true>(const EncodeCall&);
extern template void launch_encode_rows<256, true>(const EncodeCall&);
extern template void launch_encode_rows<128, true>(const EncodeCall&);
extern template void launch_dequant_rows<64, true>(const DequantCall&);
extern template void launch_dequant_rows<256, true>(const DequantCall&);
extern template void launch_dequant_rows<128, true>(const DequantCall&);
extern template void launch_encode_indices<64>(const EncodeCall&);
extern template void launch_encode_indices<128>(const EncodeCall&);
extern template void launch_encode_indices<256>(const EncodeCall&);
extern template void launch_dequant_indices<64>(const DequantCall&, uint32_t);
extern template void launch_dequant_indices<128>(const DequantCall&, uint32_t);
extern template void launch_dequant_indices<256>(const DequantCall&, uint32_t);

}  // namespace tqc
