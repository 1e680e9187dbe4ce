// Fused decode tile on the matrix cores at float32 fidelity for the head dimensions 64 and 256 (packed or fp16 keys, packed
// values of 1 to 4 bits, any number of query heads per kv head).  Included by tq_attn.hip, whose DecodeArgs, tiles of 256
// positions and merge pass it shares with the vector kernel that it stands in for.
//
// The vector kernel decodes every element for eight heads with multiply-adds: its time is vector arithmetic (2 sequences x
// 32 / 8 heads x 8 190 positions of d = 64 at four bits: 20.4 us for 9 MB; this kernel, query rotation included, 10.2).  Here a wave's 64 positions and 16 heads are
// products of 16x16x32 matrix instructions.  Operands keep 22 bits: queries, weights and centroids enter as an fp16 value and
// the fp16 remainder of its rounding, keys in fp16 are exact; queries and, in each wave, weights times value norms are scaled per
// head by powers of two, so that magnitudes outside the range of fp16 change nothing, nor does a head whose value norms lie many
// octaves below another's (see tq_split_mfma.h).  Infinite keys and queries give the infinite scores of the vector kernel, infinite
// value norms its infinite sums: a remainder never meets them.
#pragma once

// query heads of a kv head that one workgroup serves: at d = 256 eight, whose sums leave room for three workgroups in a CU's LDS
// (4 sequences x 32 / 8 heads x 16 000 positions, fp16 keys: a call takes 150 us with one workgroup of sixteen heads a CU, 84 us with three of eight)
template <int D> constexpr int kSplitHeads = D == 256 ? 8 : 16;

// power of two that brings `largest` to [2^13, 2^14), and its inverse: normal for every float (a largest below 2^-113 stays as
// many octaves below)
__device__ __forceinline__ void split_scale(float largest, float& up, float& down) {
  const int ex = min(max((int)((__float_as_uint(largest) >> 23) & 0xFF), 14), 254);
  up = __uint_as_float((uint32_t)(254 - ex + 13) << 23);
  down = __uint_as_float((uint32_t)(ex - 13) << 23);
}

// grid = (n_tiles_max, n_kv * n_rgroups, n_seq), 256 threads
template <int D, int BITS, bool DENSE>
__global__ __launch_bounds__(kThreads) void split_decode_kernel(DecodeArgs a, int q_dtype, Codebook kcb, Codebook vcb) {
  using tqm::f4;
  using tqm::h8;
  using tqm::u4;
  using VF = tqm::VField<BITS>;
  constexpr int PD = Pk<BITS>::pdim(D), PSTR = PD | 1, VPW = Pk<BITS>::VPW;
  constexpr int kH = kSplitHeads<D>;
  constexpr int KB = D / 32;                                   // contraction steps of a score
  constexpr int EL = D >= 128 ? 8 : D / 16;                    // consecutive elements of a value row per lane and pass
  constexpr int NP = D / (16 * EL);
  constexpr int EPL = D / 64;
  constexpr int kRows = 64 * PSTR + 4;                         // a field's second word may lie past the last row
  constexpr int kQ = D / 2 + 4;                                // words per query row, rows in different banks
  constexpr int kWaveWords = (DENSE ? 1 : 2) * kRows > kH * D ? (DENSE ? 1 : 2) * kRows : kH * D;
  constexpr int kLutN = VF::kLut < 64 ? 64 : VF::kLut;
  constexpr float kLog2eF = 1.44269504088896340736f;
  __shared__ __align__(16) uint32_t area_s[kWaves][(kWaveWords + 3) & ~3];   // per wave: packed rows, then its sums [16][D]
  __shared__ __align__(16) uint32_t qh_s[kH][kQ], ql_s[kH][kQ];
  __shared__ float qdown_s[kH];
  __shared__ __align__(16) uint2 lutk_s[DENSE ? 1 : kLutN], lutv_s[kLutN];
  __shared__ __align__(16) float kn_s[kWaves][64], vn_s[kWaves][64];
  __shared__ float m_s[kWaves][16], l_s[kWaves][16];

  const int tile = blockIdx.x;
  const int kvh = blockIdx.y / a.n_rgroups;
  const int r0 = (blockIdx.y % a.n_rgroups) * kH;
  const int n_local = min(kH, a.n_rep - r0);
  const int seq = blockIdx.z;
  const int n_q = a.n_kv * a.n_rep;
  const int64_t q_row0 = (int64_t)seq * n_q + (int64_t)kvh * a.n_rep + r0;
  int64_t first, len;
  seq_range(a.seq_offsets, a.seq_len, seq, first, len);
  const int64_t p0 = (int64_t)tile * kTile;
  if (p0 >= len) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n16 = lane & 15, g = lane >> 4;
  const int64_t w0 = p0 + wave * 64;                            // first position of the wave
  const int rows = (int)max((int64_t)0, min((int64_t)64, len - w0));   // uniform over the wave
  const int64_t krow0 = (int64_t)seq * a.k_seq_stride + (int64_t)kvh * a.k_head_stride + first;
  const int64_t vrow0 = (int64_t)seq * a.v_seq_stride + (int64_t)kvh * a.v_head_stride + first + w0;

  // ---- packed rows and norms of the wave, query rows, tables
  uint32_t* krows = area_s[wave];
  uint32_t* vrows = area_s[wave] + (DENSE ? 0 : kRows);
  const int last = rows > 0 ? rows * PD - 1 : 0;                // every load is of a word that exists: no branch around one
  const uint32_t* ksrc = DENSE ? nullptr : a.k_packed + (krow0 + (rows > 0 ? w0 : p0)) * PD;
  const uint32_t* vsrc = a.v_packed + (vrow0 - (rows > 0 ? 0 : w0 - p0)) * PD;
  uint32_t kraw[DENSE ? 1 : PD], vraw[PD];
#pragma unroll
  for (int i = 0; i < PD; ++i) {
    const int idx = min(i * 64 + lane, last);
    if (!DENSE) kraw[i] = ksrc[idx];
    vraw[i] = vsrc[idx];
  }
  float my_kn = 0.0f, my_vn = 0.0f;
  if (lane < rows) {
    if (!DENSE) my_kn = a.k_norms[(int64_t)seq * a.kn_seq_stride + (int64_t)kvh * a.kn_head_stride + first + w0 + lane];
    my_vn = a.v_norms[(int64_t)seq * a.vn_seq_stride + (int64_t)kvh * a.vn_head_stride + first + w0 + lane];
  }
  const bool rotate = !DENSE && a.k_signs;                      // the query itself: q * signs and the butterfly of tq_prerotate_query
  float v[kH / kWaves][EPL];
#pragma unroll
  for (int it = 0; it < kH / kWaves; ++it) {
    const int r = wave + it * kWaves;
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      v[it][i] = 0.0f;
      if (r < n_local) {
        const int64_t at = (q_row0 + r) * D + lane + 64 * i;
        if (q_dtype == TQ_F32) v[it][i] = reinterpret_cast<const float*>(a.q)[at];
        else if (q_dtype == TQ_F16) v[it][i] = __half2float(reinterpret_cast<const __half*>(a.q)[at]);
        else v[it][i] = __bfloat162float(reinterpret_cast<const __hip_bfloat16*>(a.q)[at]);
        if (rotate) v[it][i] *= a.k_signs[lane + 64 * i];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < PD; ++i) {
    const int idx = i * 64 + lane, row = idx / PD;
    if (!DENSE) krows[row * PSTR + (idx - row * PD)] = kraw[i];
    vrows[row * PSTR + (idx - row * PD)] = vraw[i];
  }
  if (!DENSE) kn_s[wave][lane] = my_kn;
  vn_s[wave][lane] = my_vn;
#pragma unroll
  for (int it = 0; it < kH / kWaves; ++it) {
    const int r = wave + it * kWaves;
    if (rotate && r < n_local) raw_butterfly<D>(v[it], lane);   // uniform over the wave
    float largest = 0.0f;
#pragma unroll
    for (int i = 0; i < EPL; ++i) largest = fmaxf(largest, fabsf(v[it][i]));
    float up, down;
    split_scale(wave_max(largest), up, down);
    if (lane == 0) qdown_s[r] = down;
    __half* hi = reinterpret_cast<__half*>(&qh_s[r][0]);
    __half* lo = reinterpret_cast<__half*>(&ql_s[r][0]);
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      const float x = v[it][i] * up;
      const __half h = __float2half_rn(x);
      hi[lane + 64 * i] = h;
      lo[lane + 64 * i] = __float2half_rn(fabsf(x) == INFINITY ? 0.0f : x - __half2float(h));
    }
  }
  // fp16 keys: row n16 of a group of 16 positions, one group ahead of its products (rows past the end: the last that exists)
  u4 kd[2][DENSE ? KB : 1];
  auto load_keys = [&](int t, u4 (&k)[DENSE ? KB : 1]) {
    if constexpr (DENSE) {
      const int64_t row = krow0 + (rows > 0 ? w0 + min(16 * t + n16, rows - 1) : p0);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) k[kb] = *reinterpret_cast<const u4*>(a.k_dense + row * D + 8 * g + 32 * kb);
    }
  };
  load_keys(0, kd[0]);
  if (!DENSE && wave == 0) tqm::fill_split_table<BITS>(lutk_s, kcb, lane);
  if (wave == 1) tqm::fill_split_table<BITS>(lutv_s, vcb, lane);
  __syncthreads();

  // ---- scores: lane (head n16, group g) gets positions 16 t + 4 g + j
  u4 qh[KB], ql[KB];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    qh[kb] = *reinterpret_cast<const u4*>(&qh_s[n16 & (kH - 1)][16 * kb + 4 * g]);
    ql[kb] = *reinterpret_cast<const u4*>(&ql_s[n16 & (kH - 1)][16 * kb + 4 * g]);
  }
  const float qdown = qdown_s[n16 & (kH - 1)];      // columns past the last head repeat others and are dropped
  float s[4][4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    f4 acc = {0.f, 0.f, 0.f, 0.f}, rem = {0.f, 0.f, 0.f, 0.f};   // products of the values, products with a remainder
    if constexpr (DENSE) {
      u4 (&k)[KB] = kd[t & 1];
      if (t < 3) load_keys(t + 1, kd[(t + 1) & 1]);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        rem = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, k[kb]), __builtin_bit_cast(h8, ql[kb]), rem, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, k[kb]), __builtin_bit_cast(h8, qh[kb]), acc, 0, 0, 0);
      }
    } else {
      const uint32_t* krow = krows + (16 * t + n16) * PSTR;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int e0 = 32 * kb + 8 * g, w = e0 / VPW, sh = (e0 % VPW) * BITS;
        const uint32_t f = VF::field_raw(krow + w, sh, 30 - sh);
        u4 kh, kl;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint2 e = lutk_s[VF::index(f, k)];
          kh[k] = e.x;
          kl[k] = e.y;
        }
        rem = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, kl), __builtin_bit_cast(h8, qh[kb]), rem, 0, 0, 0);
        rem = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, kh), __builtin_bit_cast(h8, ql[kb]), rem, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, kh), __builtin_bit_cast(h8, qh[kb]), acc, 0, 0, 0);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = 16 * t + 4 * g + j;
      // an infinite key times a remainder of 0 is no number: the product of the values is the score then
      float x = (fabsf(acc[j]) == INFINITY ? acc[j] : acc[j] + rem[j]) * qdown;
      if (!DENSE) x = (x * a.k_table * kn_s[wave][row]) * a.inv_dim;
      x *= a.attn_scale;
      if (row < rows) {
        if (a.mask && n16 < n_local)
          x += a.mask[(int64_t)seq * a.mask_seq_stride + ((int64_t)kvh * a.n_rep + r0 + n16) * a.mask_head_stride + w0 + row];
      } else {
        x = -INFINITY;
      }
      s[t][j] = x;
    }
  }
  // ---- the wave's softmax: maximum, weights times value norms as value and remainder, sum of weights
  float m = -INFINITY;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) m = fmaxf(m, s[t][j]);
  m = max_over_rows(m);
  float l = 0.0f, largest = 0.0f;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float p = (m == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f((s[t][j] - m) * kLog2eF);
      l += p;
      s[t][j] = p * vn_s[wave][16 * t + 4 * g + j];
      if (n16 >= n_local) s[t][j] = 0.0f;                       // the rows past the last head hold no query
      largest = fmaxf(largest, fabsf(s[t][j]));
    }
  l = sum_over_rows(l);
  float up, down;
  largest = max_over_rows(largest);                             // of head n16
  split_scale(largest, up, down);
  if (__any(largest == INFINITY)) {                             // infinite value norms: the sign of the sum, times infinity
    if (largest == INFINITY) {
      up = 1.0f;
      down = INFINITY;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) s[t][j] = fabsf(s[t][j]) == INFINITY ? copysignf(16384.0f, s[t][j]) : s[t][j] * 0.0f;
    }
  }
  u4 ph[2], pl[2];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    float hi[4], lo[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float x = s[t][j] * up;
      hi[j] = __half2float(__float2half_rn(x));
      lo[j] = x - hi[j];
    }
    ph[t >> 1][2 * (t & 1)] = pack_h2(hi[0], hi[1]);
    ph[t >> 1][2 * (t & 1) + 1] = pack_h2(hi[2], hi[3]);
    pl[t >> 1][2 * (t & 1)] = pack_h2(lo[0], lo[1]);
    pl[t >> 1][2 * (t & 1) + 1] = pack_h2(lo[2], lo[3]);
  }
  // ---- values: lane (element group n16) of a pass decodes elements EL (n16 + 16 pass) .. of eight positions per product
  f4 acc[NP][EL];
#pragma unroll
  for (int np = 0; np < NP; ++np) {
    const int e0 = EL * (n16 + 16 * np), w = e0 / VPW, sh = (e0 % VPW) * BITS;
#pragma unroll
    for (int et = 0; et < EL; ++et) acc[np][et] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb2 = 0; kb2 < 2; ++kb2) {
      uint32_t VI[8];
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const uint32_t* ra = vrows + (16 * (2 * kb2 + (qd >> 1)) + 4 * g + 2 * (qd & 1)) * PSTR + w;
        uint32_t fa, fb;
        if constexpr (BITS == 3 || BITS * EL == 32) {
          fa = VF::field_raw(ra, sh, 30 - sh);
          fb = VF::field_raw(ra + PSTR, sh, 30 - sh);
        } else {                                                // a piece is part of one word
          fa = ra[0] >> sh;
          fb = ra[PSTR] >> sh;
        }
        VF::interleave_raw(fa, fb, VI[qd], VI[4 + qd]);
      }
#pragma unroll
      for (int et = 0; et < EL; ++et) {
        u4 bh, bl;
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          const uint2 e = lutv_s[VF::index(VI[(et & 1) * 4 + qd], et >> 1)];
          bh[qd] = e.x;
          bl[qd] = e.y;
        }
        acc[np][et] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, pl[kb2]), __builtin_bit_cast(h8, bh), acc[np][et], 0, 0, 0);
        acc[np][et] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, ph[kb2]), __builtin_bit_cast(h8, bl), acc[np][et], 0, 0, 0);
        acc[np][et] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, ph[kb2]), __builtin_bit_cast(h8, bh), acc[np][et], 0, 0, 0);
      }
    }
  }
  // ---- the wave's sums into its own area (its packed rows have been consumed), then the four waves together
  wave_lds_fence();
  float* dep = reinterpret_cast<float*>(area_s[wave]);
  float unscale[4];                                             // of heads 4 g + j, whose sums this lane holds
#pragma unroll
  for (int j = 0; j < 4; ++j) unscale[j] = __shfl(down, 4 * g + j) * a.v_table;
#pragma unroll
  for (int np = 0; np < NP; ++np)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e4 = 0; e4 < EL; e4 += 4)
        if (kH == 16 || 4 * g + j < kH) *reinterpret_cast<f4*>(dep + (4 * g + j) * D + EL * (n16 + 16 * np) + e4) =
            f4{acc[np][e4][j], acc[np][e4 + 1][j], acc[np][e4 + 2][j], acc[np][e4 + 3][j]} * unscale[j];
  if (g == 0) {
    m_s[wave][n16] = m;
    l_s[wave][n16] = l;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < n_local * (D / 4); i += kThreads) {
    const int r = i / (D / 4), e = 4 * (i % (D / 4));
    float M = m_s[0][r];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) M = fmaxf(M, m_s[w][r]);
    f4 v = {0.f, 0.f, 0.f, 0.f};
    float L = 0.0f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float mw = m_s[w][r];
      const float f = (mw == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f((mw - M) * kLog2eF);
      v += *reinterpret_cast<const f4*>(reinterpret_cast<const float*>(area_s[w]) + r * D + e) * f;
      L += l_s[w][r] * f;
    }
    const int64_t at = (q_row0 + r) * a.n_tiles_max + tile;
    *reinterpret_cast<f4*>(a.ws_S + at * D + e) = v;
    if (e == 0) {
      a.ws_ml[2 * at] = M;
      a.ws_ml[2 * at + 1] = L;
    }
  }
}
