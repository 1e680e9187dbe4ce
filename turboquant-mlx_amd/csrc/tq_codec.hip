// PolarQuant codec kernels for gfx950: fused encode, dequantise, query pre-rotation and the
// per-row-butterfly QK scoring.  One wavefront owns one vector; the Walsh-Hadamard butterfly
// and the norm reduction run on lane exchanges, never through LDS barriers.
#include "tq_codec_stream.h"

#include <math.h>
#include <algorithm>
#include <cmath>
#include <string.h>
#include <mutex>

namespace {

using namespace tqd;
using namespace tqc;

// Optional row copies done by the wavefront that encodes a row (the append of a cache that keeps
// float16 keys beside its packed values): key row `row` of k_src (dtype k_dtype) goes, converted to
// float16, to k_dst + (g * k_group_stride + r) * D, and the value row itself, unchanged, to
// v_dst + (g * v_group_stride + r) * D.  Null destinations switch a copy off.
// With pos_dev set, every destination row index (packed words, norms and the two copies) is
// shifted by the value pos_dev points to, read on the GPU when the kernel runs: a launch recorded
// once (HIP graph) then inserts at whatever position the device counter holds.  Rows that would
// land outside 0 .. pos_cap - 1 are not stored.
struct RowCopy {
  const void* k_src;
  __half* k_dst;
  void* v_dst;
  int64_t k_group_stride, v_group_stride;
  int k_dtype;
  const int64_t* pos_dev;
  int64_t pos_cap;
};

// ---------------------------------------------------------------- encode
// Per vector: sum of squares in stride-halving tree order, sqrt, divide by max(n, 1e-8), sign
// flip, raw butterfly, count of thresholds exceeded (strict >), pack.  `thr` holds the decision
// thresholds in the domain of the raw butterfly output (see encode_thresholds below).
template <int D, int BITS, typename T>
__global__ __launch_bounds__(kBlock) void encode_kernel(EncodeSides sides, Thresholds thr, RowMap rm, RowCopy rc) {
  const T* __restrict__ x = (const T*)sides.s[blockIdx.y].x;
  const float* __restrict__ signs = sides.s[blockIdx.y].signs;
  uint32_t* __restrict__ packed = sides.s[blockIdx.y].packed;
  float* __restrict__ norms = sides.s[blockIdx.y].norms;
  constexpr int EPL = Lay<D>::EPL;
  constexpr int VPW = Pk<BITS>::VPW;
  constexpr int PDIM = Pk<BITS>::pdim(D);
  constexpr int NB = (1 << BITS) - 1;
  __shared__ uint8_t idx_s[kWavesPerBlock][D >= 64 ? D : 64];

  const int lane = threadIdx.x & (TQ_WAVE - 1);
  const int wave = threadIdx.x >> 6;
  float sg[EPL];
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    int e = lane + 64 * i;
    sg[i] = (e < D) ? signs[e] : 0.0f;
  }
  const int64_t rows_per_sweep = (int64_t)gridDim.x * kWavesPerBlock;
  const int64_t n_iter = (rm.n_rows + rows_per_sweep - 1) / rows_per_sweep;
  for (int64_t it = 0; it < n_iter; ++it) {
    const int64_t row = (it * gridDim.x + blockIdx.x) * kWavesPerBlock + wave;
    const bool valid = row < rm.n_rows;
    float xv[EPL], sq[EPL];
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      int e = lane + 64 * i;
      xv[i] = (valid && e < D) ? load_as_float<T>(x + row * D + e) : 0.0f;
      sq[i] = xv[i] * xv[i];
    }
    const float ss = tree_sum<D>(sq);
    const float nrm = sqrtf(ss);
    const float safe = fmaxf(nrm, 1e-8f);
    float v[EPL];
#pragma unroll
    for (int i = 0; i < EPL; ++i) v[i] = (xv[i] / safe) * sg[i];
    raw_butterfly<D>(v, lane);
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      uint32_t idx = 0;
#pragma unroll
      for (int b = 0; b < NB; ++b) idx += (v[i] > thr.t[b]) ? 1u : 0u;
      int e = lane + 64 * i;
      if (e < D) idx_s[wave][e] = (uint8_t)idx;
    }
    __syncthreads();
    if (valid) {
      const int64_t g = row / rm.rows_per_group;
      int64_t r = row - g * rm.rows_per_group;
      bool store = true;
      if (rc.pos_dev) {
        r += *rc.pos_dev;
        store = r >= 0 && r < rc.pos_cap;
      }
      if (store) {
      if (lane < PDIM) {
        uint32_t word = 0;
#pragma unroll
        for (int i = 0; i < VPW; ++i) {
          int e = lane * VPW + i;
          if (e < D) word |= (uint32_t)idx_s[wave][e] << (i * BITS);
        }
        packed[(g * rm.packed_group_stride + r) * PDIM + lane] = word;
      }
      if (lane == 0) norms[g * rm.norms_group_stride + r] = nrm;
      if (rc.v_dst) {
        T* vd = (T*)rc.v_dst + (g * rc.v_group_stride + r) * D;
#pragma unroll
        for (int i = 0; i < EPL; ++i) {
          const int e = lane + 64 * i;
          if (e < D) vd[e] = x[row * D + e];
        }
      }
      if (rc.k_dst) {
        __half* kd = rc.k_dst + (g * rc.k_group_stride + r) * D;
#pragma unroll
        for (int i = 0; i < EPL; ++i) {
          const int e = lane + 64 * i;
          if (e < D) {
            const int64_t at = row * D + e;
            if (rc.k_dtype == TQ_F16) kd[e] = ((const __half*)rc.k_src)[at];
            else if (rc.k_dtype == TQ_F32) kd[e] = __float2half_rn(((const float*)rc.k_src)[at]);
            else kd[e] = __float2half_rn(__bfloat162float(((const __hip_bfloat16*)rc.k_src)[at]));
          }
        }
      }
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------- dequant
template <int D, int BITS>
__device__ __forceinline__ void load_centroid_values(const uint32_t* __restrict__ prow, const float* cb,
                                                     int lane, float s, float (&v)[Lay<D>::EPL]) {
  constexpr int EPL = Lay<D>::EPL;
  constexpr int VPW = Pk<BITS>::VPW;
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    int e = lane + 64 * i;
    float val = 0.0f;
    if (e < D) {
      uint32_t word = prow[e / VPW];
      uint32_t idx = (word >> ((e % VPW) * BITS)) & Pk<BITS>::MASK;
      val = cb[idx] * s;
    }
    v[i] = val;
  }
}

template <int D, int BITS, typename TO>
__global__ __launch_bounds__(kBlock) void dequant_kernel(DequantSides sides, Codebook cbk, float s, RowMap rm) {
  const uint32_t* __restrict__ packed = sides.s[blockIdx.y].packed;
  const float* __restrict__ norms = sides.s[blockIdx.y].norms;
  const float* __restrict__ signs = sides.s[blockIdx.y].signs;
  TO* __restrict__ out = (TO*)sides.s[blockIdx.y].out;
  constexpr int EPL = Lay<D>::EPL;
  constexpr int PDIM = Pk<BITS>::pdim(D);
  __shared__ float cb[16];
  if (threadIdx.x < 16) cb[threadIdx.x] = cbk.c[threadIdx.x];
  __syncthreads();
  const int lane = threadIdx.x & (TQ_WAVE - 1);
  const int wave = threadIdx.x >> 6;
  float sg[EPL];
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    int e = lane + 64 * i;
    sg[i] = (e < D) ? signs[e] : 0.0f;
  }
  const int64_t rows_per_sweep = (int64_t)gridDim.x * kWavesPerBlock;
  for (int64_t row = (int64_t)blockIdx.x * kWavesPerBlock + wave; row < rm.n_rows; row += rows_per_sweep) {
    const int64_t g = row / rm.rows_per_group;
    const int64_t r = row - g * rm.rows_per_group;
    const uint32_t* prow = packed + (g * rm.packed_group_stride + r) * PDIM;
    const float nrm = norms[g * rm.norms_group_stride + r];
    float v[EPL];
    load_centroid_values<D, BITS>(prow, cb, lane, s, v);
    raw_butterfly<D>(v, lane);
    TO* orow = out + (g * rm.out_group_stride + r) * D;
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      int e = lane + 64 * i;
      if (e < D) store_from_float<TO>(orow + e, ((v[i] * s) * sg[i]) * nrm);
    }
  }
}

// ---------------------------------------------------------------- prerotate query
template <int D, typename T>
__global__ __launch_bounds__(kBlock) void prerotate_kernel(const T* __restrict__ q,
                                                           const float* __restrict__ signs,
                                                           float* __restrict__ q_rot, int64_t n_heads) {
  constexpr int EPL = Lay<D>::EPL;
  const int lane = threadIdx.x & (TQ_WAVE - 1);
  const int wave = threadIdx.x >> 6;
  const int64_t h = (int64_t)blockIdx.x * kWavesPerBlock + wave;
  if (h >= n_heads) return;
  float v[EPL];
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    int e = lane + 64 * i;
    v[i] = (e < D) ? load_as_float<T>(q + h * D + e) * signs[e] : 0.0f;
  }
  raw_butterfly<D>(v, lane);
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    int e = lane + 64 * i;
    if (e < D) q_rot[h * D + e] = v[i];
  }
}

// ---------------------------------------------------------------- per-row-butterfly QK scores (MHA)
template <int D, int BITS>
__global__ __launch_bounds__(kBlock) void packed_qk_kernel(const float* __restrict__ query,
                                                           const uint32_t* __restrict__ packed,
                                                           const float* __restrict__ norms, Codebook cbk,
                                                           const float* __restrict__ signs, float s,
                                                           float* __restrict__ scores, int64_t seq_len,
                                                           int64_t p_head_stride, int64_t n_head_stride) {
  constexpr int EPL = Lay<D>::EPL;
  constexpr int PDIM = Pk<BITS>::pdim(D);
  __shared__ float cb[16];
  if (threadIdx.x < 16) cb[threadIdx.x] = cbk.c[threadIdx.x];
  __syncthreads();
  const int lane = threadIdx.x & (TQ_WAVE - 1);
  const int wave = threadIdx.x >> 6;
  const int head = blockIdx.y;
  float sg[EPL], qv[EPL];
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    int e = lane + 64 * i;
    sg[i] = (e < D) ? signs[e] : 0.0f;
    qv[i] = (e < D) ? query[(int64_t)head * D + e] : 0.0f;
  }
  const int64_t sweep = (int64_t)gridDim.x * kWavesPerBlock;
  for (int64_t pos = (int64_t)blockIdx.x * kWavesPerBlock + wave; pos < seq_len; pos += sweep) {
    const uint32_t* prow = packed + ((int64_t)head * p_head_stride + pos) * PDIM;
    const float nrm = norms[(int64_t)head * n_head_stride + pos];
    float v[EPL];
    load_centroid_values<D, BITS>(prow, cb, lane, s, v);
    raw_butterfly<D>(v, lane);
    float part[EPL];
#pragma unroll
    for (int i = 0; i < EPL; ++i) part[i] = (((v[i] * s) * sg[i]) * nrm) * qv[i];
    const float tot = tree_sum<D>(part);
    if (lane == 0) scores[(int64_t)head * seq_len + pos] = tot;
  }
}

// ---------------------------------------------------------------- host helpers

// order-preserving map float <-> uint32 for bisection over all finite floats
inline uint32_t f2ord(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
inline float ord2f(uint32_t o) {
  uint32_t u = (o & 0x80000000u) ? (o & 0x7FFFFFFFu) : ~o;
  float f;
  memcpy(&f, &u, 4);
  return f;
}

// The pure-array quantiser compares z = fl(fl(w*s)/s) with each boundary b, w being the raw
// butterfly output and s = float32(1/sqrt(dim)).  z is a non-decreasing function of w, so
// {w : z(w) > b} = {w : w > t} with t the largest float whose z is <= b; t is found by
// bisection over the ordered floats.  Comparing w with t gives the same index for every w,
// NaN included (both comparisons are false), without the multiply and divide per element.
float double_rounding_threshold(float b, float s) {
  auto z_le_b = [&](float w) {
    volatile float y = w * s;
    volatile float z = y / s;
    return z <= b;
  };
  uint32_t lo = f2ord(-3.4028234663852886e38f), hi = f2ord(3.4028234663852886e38f);
  if (!z_le_b(ord2f(lo))) return -INFINITY;
  if (z_le_b(ord2f(hi))) return ord2f(hi);
  while (hi - lo > 1) {  // invariant: z(lo) <= b < z(hi)
    uint32_t mid = lo + (hi - lo) / 2;
    if (z_le_b(ord2f(mid))) lo = mid; else hi = mid;
  }
  return ord2f(lo);
}

// Finds alpha, beta with  j + 1/16 < alpha * t[j] + beta < j + 1 - 1/16  for every threshold j (and a
// further margin of 0.01), beta a multiple of 1/8.  The kernel evaluates v = fma(w, alpha, beta + 2^20 + 32)
// in float: one rounding, to a multiple of 1/8, i.e. at most 1/16 away from alpha*w + beta, so
// floor(v) - 2^20 - 32 is the count of thresholds below w or one less for every w.  |w| <= sqrt(128)
// (raw butterfly of a unit vector; up to d = 128), so the guess must stay within +-32 of zero for the 64-entry table
// (three bits).  At d = 256 |w| reaches 16 and the kernel clamps to the table's first and last cell: every threshold
// must then lie in a cell of the table (here they lie in cells 0 .. nb - 1).
// False when no such line exists (then the generic kernel counts the thresholds one by one).
bool level_guess_search(const float* t, int nb, EncodeGuess& out);

// Widths other than three bits: any line u = alpha * t + beta0 (beta0 a multiple of 1/8) under which no cell
// [c, c + 1) of u holds two thresholds and every threshold keeps the margin above from both edges of its cell.
// The kernel's cell of w is floor(alpha * w + beta0) or, for w within 1/16 below a cell edge, the next one; with no
// threshold that close below an edge the count "thresholds below the cell + (w > the threshold inside it)" is the
// count of thresholds below w either way.  The candidate with the widest margin is taken.
// A threshold below the table's first cell refuses the line: no number reaches it, but an output that is no number (a row with
// an infinity) reads the first cell, whose count must be 0.  clamped (d = 256): one above the last cell does as well.
bool level_cells_search(const float* t, int nb, bool clamped, EncodeGuess& out) {
  for (int i = 0; i < nb; ++i)
    if (!std::isfinite(t[i]) || (i > 0 && !(t[i] > t[i - 1]))) return false;
  const int half = nb == 15 ? 64 : 32;                              // the kernel's table has 2 * half cells
  const double margin = 1.0 / 16.0 + 0.01;
  double best = -1.0, best_b = 0.0;
  float best_a = 0.0f;
  for (int ai = 4000; ai >= 100; --ai) {
    const float af = (float)(ai * ((half - 1) / 11.4 / 4000.0));    // up to (half - 1) / 11.4 cells per unit of w
    const double a = (double)af;
    for (int bi = -64; bi <= 64; ++bi) {
      const double b = bi / 8.0;
      if (!(a * 11.4 + std::fabs(b) < half - 1.0)) continue;
      double slack = 1e9, prev_cell = -1e9;
      bool ok = true;
      for (int j = 0; j < nb && ok; ++j) {
        const double u = a * (double)t[j] + b;
        const double c = std::floor(u), f = u - c;
        if (f < margin || f > 1.0 - margin || c <= prev_cell || c < -half || (clamped && c > half - 1)) ok = false;
        prev_cell = c;
        slack = std::fmin(slack, std::fmin(f - margin, 1.0 - margin - f));
      }
      if (ok && slack > best) { best = slack; best_a = af; best_b = b; }
    }
    if (best > 0.15) break;                                         // good enough: finer cells gain nothing
  }
  if (best < 0.0) return false;
  out.alpha = best_a;
  out.beta0 = (float)best_b;
  out.beta = (float)(best_b + 1048576.0 + (double)half);            // exact: a multiple of 1/8 below 2^21
  return true;
}

// Thresholds and level guess of the encoder for the last few (boundaries, dim, variant) seen, by value: a process that
// alternates widths or threshold rules between calls -- caches of different bits, keys and values under different
// rules -- would otherwise repeat the search for a guess at every switch, and every call the bisections of
// double_rounding_threshold (2 us at three bits).  The search (0.3 ms at three bits, 13 ms at four) is made for callers
// that use the guess only: a token's step never waits for it.  The lock covers the table only, not the search: two
// threads that miss on the same set both search and store the same result.
struct EncodePlan {
  Thresholds thr;
  EncodeGuess gs;
  bool has_guess;
};

EncodePlan encode_plan(const float* boundaries, int dim, int bits, int variant, bool want_guess) {
  constexpr int kSlots = 32;                                         // every width, head dimension and rule there is, and a few given tables
  struct Slot { float b[15]; int nb, dim, variant; bool searched; EncodePlan p; };
  static std::mutex mu;
  static Slot slots[kSlots];
  static int n_used = 0, next = 0;
  const int nb = (1 << bits) - 1;
  auto find = [&]() -> Slot* {                                        // under the lock
    for (int i = 0; i < n_used; ++i)
      if (slots[i].nb == nb && slots[i].dim == dim && slots[i].variant == variant &&
          memcmp(slots[i].b, boundaries, nb * sizeof(float)) == 0)
        return &slots[i];
    return nullptr;
  };
  Slot s{};
  bool known = false;
  {
    std::lock_guard<std::mutex> lock(mu);
    if (const Slot* hit = find()) {
      if (hit->searched || !want_guess) return hit->p;
      s = *hit;
      known = true;
    }
  }
  if (!known) {
    s.nb = nb;
    s.dim = dim;
    s.variant = variant;
    memcpy(s.b, boundaries, nb * sizeof(float));
    for (int i = 0; i < 15; ++i) s.p.thr.t[i] = INFINITY;
    tq::encode_thresholds(boundaries, dim, bits, variant, s.p.thr.t);
  }
  if (want_guess) {
    s.p.has_guess = (nb == 7) ? level_guess_search(s.p.thr.t, nb, s.p.gs) : level_cells_search(s.p.thr.t, nb, dim > 128, s.p.gs);
    s.searched = true;
  }
  {
    std::lock_guard<std::mutex> lock(mu);
    if (Slot* hit = find()) {
      if (!hit->searched) *hit = s;
    } else {
      slots[next] = s;
      next = (next + 1) % kSlots;
      if (n_used < kSlots) ++n_used;
    }
  }
  return s.p;
}

bool level_guess_search(const float* t, int nb, EncodeGuess& out) {
  for (int i = 0; i < nb; ++i)
    if (!std::isfinite(t[i]) || (i > 0 && !(t[i] > t[i - 1]))) return false;
  const double span = (double)t[nb - 1] - (double)t[0];
  if (!(span > 0)) return false;
  double best_w = 0.0, best_a = 0.0, best_b = 0.0;
  for (int s = 1; s <= 4000; ++s) {
    const double a = (double)(nb + 1) * s / (1000.0 * span);       // up to 4x the mean level density
    double lo = -1e300, hi = 1e300;
    for (int j = 0; j < nb; ++j) {
      lo = std::fmax(lo, j - a * (double)t[j]);
      hi = std::fmin(hi, j + 1 - a * (double)t[j]);
    }
    if (hi - lo > best_w) { best_w = hi - lo; best_a = a; best_b = 0.5 * (lo + hi); }
  }
  if (best_w < 0.2) return false;
  out.alpha = (float)best_a;
  const double a = (double)out.alpha;
  double lo = -1e300, hi = 1e300;
  for (int j = 0; j < nb; ++j) {
    lo = std::fmax(lo, j - a * (double)t[j]);
    hi = std::fmin(hi, j + 1 - a * (double)t[j]);
  }
  const double b = std::floor(0.5 * (lo + hi) * 8.0 + 0.5) / 8.0;
  const double margin = 1.0 / 16.0 + 0.01;
  if (!(b - lo >= margin && hi - b >= margin)) return false;
  if (!(a * 11.4 + std::fabs(b) < 31.0)) return false;
  out.beta = (float)(b + 1048576.0 + 32.0);                  // exact: a multiple of 1/8 below 2^21
  out.beta0 = (float)b;
  return true;
}

// Rows from which the streaming kernels are ahead of one wavefront per vector (encode_kernel, dequant_kernel): below,
// the chip is not full either way and the chain of a single vector spread over 64 lanes is the shorter one.  Measured on
// both sides of each line (us, streaming / one wavefront per vector; encode, then dequant to fp16):
//   d =  64:  4 097 rows 4.7 / 4.0 and 4.0 / 3.1,  16 385 rows 4.9 / 9.9 and 4.2 / 4.8,  262 147 rows 14 / 69 and 9.1 / 30
//   d = 128:  4 097 rows 4.7 / 4.3 and 4.0 / 3.4,  16 385 rows 5.4 / 11.0 and 4.5 / 5.7,  80 056 rows 9.8 / 26 and 7.7 / 14
//   d = 256:  2 049 rows 4.7 / 4.5 and 4.2 / 3.2,   8 193 rows 5.3 / 7.3 and 4.6 / 5.1,  262 147 rows 42 / 134 and 30 / 54
int64_t stream_min_rows(int dim, bool encode) {
  if (dim == 64) return encode ? 6144 : 12288;
  if (dim == 128) return encode ? 5120 : 8192;
  return encode ? 3072 : 6144;
}

RowMap row_map(int64_t n_rows, int64_t rows_per_group, int64_t packed_group_stride, int64_t norms_group_stride,
               int64_t out_group_stride) {
  RowMap rm{n_rows, rows_per_group, packed_group_stride, norms_group_stride, out_group_stride, 0, 0};
  // row / d = (row * m) >> (31 + s) with s = ceil(log2 d), m = ceil(2^(31 + s) / d), exact for row < 2^31: the error
  // row * (m d - 2^(31 + s)) stays below 2^31 * 2^s; m < 2^32 because d > 2^(s - 1)
  const uint64_t d = (uint64_t)rows_per_group;
  if (d > 1 && d < ((uint64_t)1 << 31)) {
    int s = 1;
    while (((uint64_t)1 << s) < d) ++s;
    const unsigned __int128 top = (unsigned __int128)1 << (31 + s);
    rm.group_mul = (uint32_t)((top + d - 1) / d);
    rm.group_shift = (uint32_t)(s - 1);
  }
  return rm;
}

// The streaming kernels index rows with 32 bits: rows of the call, and of the storage they lie in.
bool rows_fit_32_bits(const RowMap& rm, int64_t n_groups) {
  const int64_t most = (int64_t)1 << 31;
  return rm.n_rows < most && n_groups * rm.packed_group_stride + rm.rows_per_group < most &&
         n_groups * rm.out_group_stride + rm.rows_per_group < most;
}

// d = 128, groups of a multiple of 16 rows: the form without per-row destinations, at any size
bool whole_batches(int dim, const RowMap& rm) { return dim == 128 && rm.rows_per_group % VecLanes<128>::kVecs == 0; }

int grid_for_rows(int64_t rows) {
  int64_t blocks = (rows + kWavesPerBlock - 1) / kWavesPerBlock;
  const int64_t cap = 256 * 16;  // 16 blocks of 4 waves per CU keeps every SIMD supplied
  if (blocks > cap) blocks = cap;
  if (blocks < 1) blocks = 1;
  return (int)blocks;
}

}  // namespace

// Key and value rows of one decode step in one launch (d = 128, BITS bits, one wavefront per row): rows
// 0 .. n_rows - 1 are the keys (signs, destination 0), rows n_rows .. 2 n_rows - 1 the values.  Same
// arithmetic, operation for operation, as encode_kernel.
struct PairSide {
  const void* x;
  const float* signs;
  uint32_t* packed;
  float* norms;
  int dtype;
};

// With pos_dev set the destination row of group g is g * group_stride + *pos_dev (read when the kernel runs;
// nothing is stored when that position is outside 0 .. group_stride - 1).
template <int BITS>
__global__ __launch_bounds__(kBlock) void encode_pair_kernel(PairSide k, PairSide v, Thresholds thr, int64_t n_rows,
                                                             int64_t group_stride, const int64_t* pos_dev) {
  constexpr int D = 128, PDIM = BITS == 3 ? 13 : 4 * BITS, VPW = BITS == 3 ? 10 : 32 / BITS, NB = (1 << BITS) - 1;
  const int lane = threadIdx.x & (TQ_WAVE - 1);
  const int wave = threadIdx.x >> 6;
  const int64_t slot = (int64_t)blockIdx.x * kWavesPerBlock + wave;
  if (slot >= 2 * n_rows) return;                          // no barriers below: a wavefront may leave alone
  const bool is_v = slot >= n_rows;
  const PairSide& s = is_v ? v : k;
  const int64_t row = is_v ? slot - n_rows : slot;
  float xv[2], sq[2], sg[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int64_t at = row * D + lane + 64 * i;
    xv[i] = s.dtype == TQ_F16 ? __half2float(((const __half*)s.x)[at])
          : s.dtype == TQ_F32 ? ((const float*)s.x)[at] : __bfloat162float(((const __hip_bfloat16*)s.x)[at]);
    sg[i] = s.signs[lane + 64 * i];
    sq[i] = xv[i] * xv[i];
  }
  const float ss = tree_sum<D>(sq);
  const float nrm = sqrtf(ss);
  const float safe = fmaxf(nrm, 1e-8f);
  float w[2] = {(xv[0] / safe) * sg[0], (xv[1] / safe) * sg[1]};
  raw_butterfly<D>(w, lane);
  int idx[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint32_t n = 0;
#pragma unroll
    for (int b = 0; b < NB; ++b) n += (w[i] > thr.t[b]) ? 1u : 0u;
    idx[i] = (int)n;
  }
  uint32_t word = 0;                                       // word `lane`: elements VPW * lane .. VPW * lane + VPW - 1
#pragma unroll
  for (int i = 0; i < VPW; ++i) {
    const int e = min(VPW * lane + i, D - 1);
    const int lo = __shfl(idx[0], e & 63), hi = __shfl(idx[1], e & 63);
    const uint32_t fld = (uint32_t)((e >> 6) ? hi : lo);
    if (VPW * lane + i < D) word |= fld << (BITS * i);
  }
  int64_t dst = row * group_stride;
  if (pos_dev) {
    const int64_t pos = *pos_dev;
    if (pos < 0 || pos >= group_stride) return;
    dst += pos;
  }
  if (lane < PDIM) s.packed[dst * PDIM + lane] = word;
  if (lane == 0) s.norms[dst] = nrm;
}

namespace tq {
int encode_pair(const void* k_new, int k_dtype, const float* k_signs, uint32_t* k_packed, float* k_norms,
                const void* v_new, int v_dtype, const float* v_signs, uint32_t* v_packed, float* v_norms,
                const float* boundaries, int bits, int64_t n_rows, int64_t group_stride, int variant, tq_stream_t stream_,
                const int64_t* pos_dev) {
  const Thresholds thr = encode_plan(boundaries, 128, bits, variant, false).thr;
  PairSide k{k_new, k_signs, k_packed, k_norms, k_dtype}, v{v_new, v_signs, v_packed, v_norms, v_dtype};
  const int grid = (int)((2 * n_rows + kWavesPerBlock - 1) / kWavesPerBlock);
  TQ_DISPATCH_BITS(bits, (encode_pair_kernel<B_><<<grid, kBlock, 0, (hipStream_t)stream_>>>(k, v, thr, n_rows, group_stride, pos_dev)));
  TQ_CHECK_LAUNCH("encode_pair launch");
  return TQ_OK;
}

void encode_thresholds(const float* boundaries, int dim, int bits, int variant, float* thr_out) {
  const float s = (float)(1.0 / sqrt((double)dim));
  const int nb = (1 << bits) - 1;
  for (int i = 0; i < nb; ++i)
    thr_out[i] = (variant == TQ_ENCODE_MLX) ? double_rounding_threshold(boundaries[i], s) : boundaries[i];
}
}  // namespace tq

// ------------------------------------------------------------------ C ABI

extern "C" int tq_version(void) { return TQ_VERSION; }

extern "C" const char* tq_last_error(void) { return tq::err_buf(); }

extern "C" const char* tq_status_string(int status) {
  switch (status) {
    case TQ_OK: return "ok";
    case TQ_ERR_NULL: return "null pointer";
    case TQ_ERR_DIM: return "bad dim";
    case TQ_ERR_BITS: return "bad bits";
    case TQ_ERR_NREP: return "bad n_rep";
    case TQ_ERR_ALIGN: return "misaligned pointer";
    case TQ_ERR_DTYPE: return "bad dtype";
    case TQ_ERR_BLOCK: return "bad block_size";
    case TQ_ERR_WORKSPACE: return "workspace too small";
    case TQ_ERR_ARG: return "bad argument";
    case TQ_ERR_UNSUPPORTED: return "unsupported";
  }
  return status <= TQ_ERR_HIP ? "hip error" : "unknown";
}

namespace {
// The rows of one tensor, or of the keys and the values (n_sides = 2): arguments checked here, `who` names the entry.
int encode_sides(const char* who, const EncodeSides& sides, int n_sides, int x_dtype, const float* boundaries, int64_t n_groups,
                 int64_t rows_per_group, int64_t packed_group_stride, int64_t norms_group_stride, int dim, int bits,
                 int variant, hipStream_t stream) {
  if (int rc = tq::check_dim_bits(dim, bits)) return rc;
  if (tq::check_dtype(x_dtype)) return tq::fail(TQ_ERR_DTYPE, "%s: unknown x_dtype %d", who, x_dtype);
  if (variant != TQ_ENCODE_MLX && variant != TQ_ENCODE_METAL)
    return tq::fail(TQ_ERR_ARG, "%s: unknown variant %d", who, variant);
  if (n_groups < 0 || rows_per_group < 0) return tq::fail(TQ_ERR_ARG, "%s: negative row count", who);
  const int64_t n_rows = n_groups * rows_per_group;
  if (n_rows == 0) return TQ_OK;
  if (!boundaries) return tq::fail(TQ_ERR_NULL, "%s: null pointer", who);
  bool wide = true;                                            // 16-byte loads of the input rows
  for (int i = 0; i < n_sides; ++i) {
    const EncodeSide& s = sides.s[i];
    if (!s.x || !s.signs || !s.packed || !s.norms) return tq::fail(TQ_ERR_NULL, "%s: null pointer", who);
    if (!tq::aligned(s.x, tq::dtype_size(x_dtype)) || !tq::aligned(s.signs, 4) || !tq::aligned(s.packed, 4) ||
        !tq::aligned(s.norms, 4))
      return tq::fail(TQ_ERR_ALIGN, "%s: misaligned pointer", who);
    wide = wide && tq::aligned(s.x, 16);
  }
  const RowMap rm = row_map(n_rows, rows_per_group, packed_group_stride, norms_group_stride, 0);
  const bool whole = whole_batches(dim, rm);
  const bool stream_form = dim >= 64 && (whole || n_rows * n_sides >= stream_min_rows(dim, true)) && n_rows < (int64_t)1 << 31 &&
                           (whole || rows_fit_32_bits(rm, n_groups)) && wide;
  const EncodePlan plan = encode_plan(boundaries, dim, bits, variant, stream_form);
  if (stream_form && plan.has_guess) {
    const EncodeCall c{sides, n_sides, x_dtype, plan.thr, plan.gs, rm, bits, stream};
    if (whole) launch_encode_rows<128, false>(c);
    else if (dim == 64) launch_encode_rows<64, true>(c);
    else if (dim == 128) launch_encode_rows<128, true>(c);
    else launch_encode_rows<256, true>(c);
  } else {
    const dim3 grid(grid_for_rows(n_rows), n_sides);
#define LAUNCH_ENC(T)                                                                                                 \
    TQ_DISPATCH_DIM(dim, TQ_DISPATCH_BITS(bits, (encode_kernel<D_, B_, T><<<grid, kBlock, 0, stream>>>(                \
                                                    sides, plan.thr, rm, RowCopy{}))))
    if (x_dtype == TQ_F32) { LAUNCH_ENC(float); }
    else if (x_dtype == TQ_F16) { LAUNCH_ENC(__half); }
    else { LAUNCH_ENC(__hip_bfloat16); }
#undef LAUNCH_ENC
  }
  TQ_CHECK_LAUNCH(who);
  return TQ_OK;
}

int dequant_sides(const char* who, const DequantSides& sides, int n_sides, const float* centroids, int out_dtype,
                  int64_t n_groups, int64_t rows_per_group, int64_t packed_group_stride, int64_t norms_group_stride,
                  int64_t out_group_stride, int dim, int bits, hipStream_t stream) {
  if (int rc = tq::check_dim_bits(dim, bits)) return rc;
  if (tq::check_dtype(out_dtype)) return tq::fail(TQ_ERR_DTYPE, "%s: unknown out_dtype %d", who, out_dtype);
  if (n_groups < 0 || rows_per_group < 0) return tq::fail(TQ_ERR_ARG, "%s: negative row count", who);
  const int64_t n_rows = n_groups * rows_per_group;
  if (n_rows == 0) return TQ_OK;
  if (!centroids) return tq::fail(TQ_ERR_NULL, "%s: null pointer", who);
  bool wide = (out_group_stride * dim * (int64_t)tq::dtype_size(out_dtype)) % 16 == 0;   // 16-byte stores of the output rows
  for (int i = 0; i < n_sides; ++i) {
    const DequantSide& s = sides.s[i];
    if (!s.packed || !s.norms || !s.signs || !s.out) return tq::fail(TQ_ERR_NULL, "%s: null pointer", who);
    if (!tq::aligned(s.packed, 4) || !tq::aligned(s.norms, 4) || !tq::aligned(s.signs, 4) ||
        !tq::aligned(s.out, tq::dtype_size(out_dtype)))
      return tq::fail(TQ_ERR_ALIGN, "%s: misaligned pointer", who);
    wide = wide && tq::aligned(s.out, 16);
  }
  Codebook cb;
  for (int i = 0; i < 16; ++i) cb.c[i] = i < (1 << bits) ? centroids[i] : 0.0f;
  const float s = (float)(1.0 / sqrt((double)dim));
  const RowMap rm = row_map(n_rows, rows_per_group, packed_group_stride, norms_group_stride, out_group_stride);
  const bool whole = whole_batches(dim, rm);
  if (dim >= 64 && (whole || n_rows * n_sides >= stream_min_rows(dim, false)) && n_rows < (int64_t)1 << 31 &&
      (whole || rows_fit_32_bits(rm, n_groups)) && wide) {
    const DequantCall c{sides, n_sides, cb, s, out_dtype, rm, bits, stream};
    if (whole) launch_dequant_rows<128, false>(c);
    else if (dim == 64) launch_dequant_rows<64, true>(c);
    else if (dim == 128) launch_dequant_rows<128, true>(c);
    else launch_dequant_rows<256, true>(c);
  } else {
    const dim3 grid(grid_for_rows(n_rows), n_sides);
#define LAUNCH_DEQ(T)                                                                                                 \
    TQ_DISPATCH_DIM(dim, TQ_DISPATCH_BITS(bits, (dequant_kernel<D_, B_, T><<<grid, kBlock, 0, stream>>>(sides, cb, s, rm))))
    if (out_dtype == TQ_F32) { LAUNCH_DEQ(float); }
    else if (out_dtype == TQ_F16) { LAUNCH_DEQ(__half); }
    else { LAUNCH_DEQ(__hip_bfloat16); }
#undef LAUNCH_DEQ
  }
  TQ_CHECK_LAUNCH(who);
  return TQ_OK;
}
}  // namespace

extern "C" int tq_encode(const void* x, int x_dtype, const float* signs, const float* boundaries,
                         uint32_t* packed, float* norms, int64_t n_groups, int64_t rows_per_group,
                         int64_t packed_group_stride, int64_t norms_group_stride, int dim, int bits,
                         int variant, tq_stream_t stream_) {
  return encode_sides("tq_encode", EncodeSides{{{x, signs, packed, norms}, {}}}, 1, x_dtype, boundaries, n_groups,
                      rows_per_group, packed_group_stride, norms_group_stride, dim, bits, variant, (hipStream_t)stream_);
}

extern "C" int tq_encode_kv(const void* k, const float* k_signs, uint32_t* k_packed, float* k_norms, const void* v,
                            const float* v_signs, uint32_t* v_packed, float* v_norms, int x_dtype,
                            const float* boundaries, int64_t n_groups, int64_t rows_per_group,
                            int64_t packed_group_stride, int64_t norms_group_stride, int dim, int bits, int variant,
                            tq_stream_t stream_) {
  return encode_sides("tq_encode_kv", EncodeSides{{{k, k_signs, k_packed, k_norms}, {v, v_signs, v_packed, v_norms}}}, 2,
                      x_dtype, boundaries, n_groups, rows_per_group, packed_group_stride, norms_group_stride, dim, bits,
                      variant, (hipStream_t)stream_);
}

// Any number of rows: the launch of its own that the bytes would need costs more than one wavefront per vector saves on few rows
// (see stream_min_rows).
extern "C" int tq_quantize(const void* x, int x_dtype, const float* signs, const float* boundaries, uint8_t* indices, float* norms,
                           int64_t n_rows, int dim, int bits, int variant, tq_stream_t stream_) {
  const char* who = "tq_quantize";
  if (int rc = tq::check_dim_bits(dim, bits)) return rc;
  if (tq::check_dtype(x_dtype)) return tq::fail(TQ_ERR_DTYPE, "%s: unknown x_dtype %d", who, x_dtype);
  if (variant != TQ_ENCODE_MLX && variant != TQ_ENCODE_METAL) return tq::fail(TQ_ERR_ARG, "%s: unknown variant %d", who, variant);
  if (n_rows < 0) return tq::fail(TQ_ERR_ARG, "%s: negative row count", who);
  if (n_rows == 0) return TQ_OK;
  if (!x || !signs || !boundaries || !indices || !norms) return tq::fail(TQ_ERR_NULL, "%s: null pointer", who);
  if (!tq::aligned(x, tq::dtype_size(x_dtype)) || !tq::aligned(signs, 4) || !tq::aligned(norms, 4))
    return tq::fail(TQ_ERR_ALIGN, "%s: misaligned pointer", who);
  if (dim < 64 || n_rows >= (int64_t)1 << 31 || !tq::aligned(x, 16) || !tq::aligned(indices, 16))
    return tq::fail(TQ_ERR_UNSUPPORTED, "%s: rows of %d, %lld of them, or a pointer off 16 bytes", who, dim, (long long)n_rows);
  const EncodePlan plan = encode_plan(boundaries, dim, bits, variant, true);
  if (!plan.has_guess) return tq::fail(TQ_ERR_UNSUPPORTED, "%s: no level line for these boundaries", who);
  const EncodeCall c{EncodeSides{{{x, signs, (uint32_t*)indices, norms}, {}}}, 1, x_dtype, plan.thr, plan.gs,
                     row_map(n_rows, n_rows, 0, 0, 0), bits, (hipStream_t)stream_};
  if (dim == 64) launch_encode_indices<64>(c);
  else if (dim == 128) launch_encode_indices<128>(c);
  else launch_encode_indices<256>(c);
  TQ_CHECK_LAUNCH(who);
  return TQ_OK;
}

extern "C" int tq_dequantize(const uint8_t* indices, const float* norms, const float* centroids, const float* signs, float* out,
                             int64_t n_rows, int dim, int bits, tq_stream_t stream_) {
  const char* who = "tq_dequantize";
  if (int rc = tq::check_dim_bits(dim, bits)) return rc;
  if (n_rows < 0) return tq::fail(TQ_ERR_ARG, "%s: negative row count", who);
  if (n_rows == 0) return TQ_OK;
  if (!indices || !norms || !centroids || !signs || !out) return tq::fail(TQ_ERR_NULL, "%s: null pointer", who);
  if (!tq::aligned(norms, 4) || !tq::aligned(signs, 4) || !tq::aligned(out, 4)) return tq::fail(TQ_ERR_ALIGN, "%s: misaligned pointer", who);
  if (dim < 64 || n_rows >= (int64_t)1 << 31 || !tq::aligned(indices, 8) || !tq::aligned(out, 16))
    return tq::fail(TQ_ERR_UNSUPPORTED, "%s: rows of %d, %lld of them, or a misaligned pointer", who, dim, (long long)n_rows);
  Codebook cb;
  for (int i = 0; i < 16; ++i) cb.c[i] = i < (1 << bits) ? centroids[i] : 0.0f;
  const RowMap rm = row_map(n_rows, n_rows, 0, 0, 0);
  const DequantCall c{DequantSides{{{(const uint32_t*)indices, norms, signs, out}, {}}}, 1, cb, (float)(1.0 / sqrt((double)dim)), TQ_F32,
                      rm, bits, (hipStream_t)stream_};
  // bytes past the width: the two upper bits of a word reach the next chunk where dequant_sides streams its words, else they do not
  const bool streams = whole_batches(dim, rm) || n_rows >= stream_min_rows(dim, false);
  const uint32_t word_bits = bits == 3 && !streams ? 0x3FFFFFFFu : ~0u;
  if (dim == 64) launch_dequant_indices<64>(c, word_bits);
  else if (dim == 128) launch_dequant_indices<128>(c, word_bits);
  else launch_dequant_indices<256>(c, word_bits);
  TQ_CHECK_LAUNCH(who);
  return TQ_OK;
}

namespace {
int vonly_append(const void* k_new, int k_dtype, const void* v_new, int v_dtype,
                               const float* v_signs, const float* boundaries, void* k_f16, void* v_raw,
                               uint32_t* v_packed, float* v_norms, int64_t n_groups, int64_t rows_per_group,
                               int64_t k_group_stride, int64_t v_raw_group_stride, int64_t packed_group_stride,
                               int64_t norms_group_stride, int dim, int bits, int variant, const int64_t* pos_dev,
                               int64_t pos_cap, tq_stream_t stream_) {
  if (int rc = tq::check_dim_bits(dim, bits)) return rc;
  if (tq::check_dtype(k_dtype) || tq::check_dtype(v_dtype))
    return tq::fail(TQ_ERR_DTYPE, "tq_vonly_append: unknown dtype %d / %d", k_dtype, v_dtype);
  if (variant != TQ_ENCODE_MLX && variant != TQ_ENCODE_METAL)
    return tq::fail(TQ_ERR_ARG, "tq_vonly_append: unknown variant %d", variant);
  if (n_groups < 0 || rows_per_group < 0) return tq::fail(TQ_ERR_ARG, "tq_vonly_append: negative row count");
  const int64_t n_rows = n_groups * rows_per_group;
  if (n_rows == 0) return TQ_OK;
  if (!k_new || !v_new || !v_signs || !boundaries || !k_f16 || !v_packed || !v_norms)
    return tq::fail(TQ_ERR_NULL, "tq_vonly_append: null pointer");
  if (!tq::aligned(k_new, tq::dtype_size(k_dtype)) || !tq::aligned(v_new, tq::dtype_size(v_dtype)) ||
      !tq::aligned(v_signs, 4) || !tq::aligned(k_f16, 2) || !tq::aligned(v_packed, 4) || !tq::aligned(v_norms, 4) ||
      (v_raw && !tq::aligned(v_raw, tq::dtype_size(v_dtype))))
    return tq::fail(TQ_ERR_ALIGN, "tq_vonly_append: misaligned pointer");
  const Thresholds thr = encode_plan(boundaries, dim, bits, variant, false).thr;
  const RowMap rm = row_map(n_rows, rows_per_group, packed_group_stride, norms_group_stride, 0);
  if (pos_dev && (!tq::aligned(pos_dev, 8) || pos_cap < 1))
    return tq::fail(TQ_ERR_ARG, "tq_vonly_append_at: position_dev must be 8-byte aligned and t_alloc >= 1");
  RowCopy rc{k_new, (__half*)k_f16, v_raw, k_group_stride, v_raw_group_stride, k_dtype, pos_dev, pos_cap};
  hipStream_t stream = (hipStream_t)stream_;
  const int grid = grid_for_rows(n_rows);
  const EncodeSides sides{{{v_new, v_signs, v_packed, v_norms}, {}}};
#define LAUNCH_APP(T)                                                                               \
  TQ_DISPATCH_DIM(dim, TQ_DISPATCH_BITS(bits, (encode_kernel<D_, B_, T><<<grid, kBlock, 0, stream>>>( \
                                                  sides, thr, rm, rc))))
  if (v_dtype == TQ_F32) { LAUNCH_APP(float); }
  else if (v_dtype == TQ_F16) { LAUNCH_APP(__half); }
  else { LAUNCH_APP(__hip_bfloat16); }
#undef LAUNCH_APP
  TQ_CHECK_LAUNCH("tq_vonly_append launch");
  return TQ_OK;
}
}  // namespace

extern "C" int tq_vonly_append(const void* k_new, int k_dtype, const void* v_new, int v_dtype,
                               const float* v_signs, const float* boundaries, void* k_f16, void* v_raw,
                               uint32_t* v_packed, float* v_norms, int64_t n_groups, int64_t rows_per_group,
                               int64_t k_group_stride, int64_t v_raw_group_stride, int64_t packed_group_stride,
                               int64_t norms_group_stride, int dim, int bits, int variant, tq_stream_t stream_) {
  return vonly_append(k_new, k_dtype, v_new, v_dtype, v_signs, boundaries, k_f16, v_raw, v_packed, v_norms, n_groups,
                      rows_per_group, k_group_stride, v_raw_group_stride, packed_group_stride, norms_group_stride, dim,
                      bits, variant, nullptr, 0, stream_);
}

extern "C" int tq_vonly_append_at(const void* k_new, int k_dtype, const void* v_new, int v_dtype,
                                  const float* v_signs, const float* boundaries, void* k_f16, void* v_raw,
                                  uint32_t* v_packed, float* v_norms, int64_t n_groups, int64_t rows_per_group,
                                  int64_t t_alloc, int dim, int bits, int variant, const int64_t* position_dev,
                                  tq_stream_t stream_) {
  if (!position_dev) return tq::fail(TQ_ERR_NULL, "tq_vonly_append_at: null position_dev");
  if (rows_per_group > t_alloc)
    return tq::fail(TQ_ERR_ARG, "tq_vonly_append_at: %lld new rows per group do not fit %lld positions",
                    (long long)rows_per_group, (long long)t_alloc);
  return vonly_append(k_new, k_dtype, v_new, v_dtype, v_signs, boundaries, k_f16, v_raw, v_packed, v_norms, n_groups,
                      rows_per_group, t_alloc, t_alloc, t_alloc, t_alloc, dim, bits, variant, position_dev, t_alloc,
                      stream_);
}

extern "C" int tq_dequant(const uint32_t* packed, const float* norms, const float* centroids,
                          const float* signs, void* out, int out_dtype, int64_t n_groups,
                          int64_t rows_per_group, int64_t packed_group_stride, int64_t norms_group_stride,
                          int64_t out_group_stride, int dim, int bits, tq_stream_t stream_) {
  return dequant_sides("tq_dequant", DequantSides{{{packed, norms, signs, out}, {}}}, 1, centroids, out_dtype, n_groups,
                       rows_per_group, packed_group_stride, norms_group_stride, out_group_stride, dim, bits,
                       (hipStream_t)stream_);
}

extern "C" int tq_dequant_kv(const uint32_t* k_packed, const float* k_norms, const float* k_signs, void* k_out,
                             const uint32_t* v_packed, const float* v_norms, const float* v_signs, void* v_out,
                             const float* centroids, int out_dtype, int64_t n_groups, int64_t rows_per_group,
                             int64_t packed_group_stride, int64_t norms_group_stride, int64_t out_group_stride, int dim,
                             int bits, tq_stream_t stream_) {
  return dequant_sides("tq_dequant_kv", DequantSides{{{k_packed, k_norms, k_signs, k_out}, {v_packed, v_norms, v_signs, v_out}}},
                       2, centroids, out_dtype, n_groups, rows_per_group, packed_group_stride, norms_group_stride,
                       out_group_stride, dim, bits, (hipStream_t)stream_);
}

// ---------------------------------------------------------------- storage set-up

namespace {
// One launch for everything that a cache's fresh storage needs besides its new rows: per segment and group, words
// 0 .. copy - 1 from the old storage, zeros in words zero_from .. zero_to - 1.
struct FillArgs {
  struct Segment {
    uint32_t* dst;
    const uint32_t* src;
    int64_t dst_stride, src_stride, copy, zero_from, zero_to, n_groups;
    int wide;                                                  // every bound a multiple of four words, 16-byte aligned
  } s[TQ_FILL_MAX_SEGMENTS];
  int n_segments;
  // behind them (blockIdx.y = n_segments): the diagonals of n_seeds seeds
  uint64_t seeds[TQ_SIGNS_MAX_SEEDS];
  int n_seeds, dim;
  float* signs;
};

template <typename V>
__device__ __forceinline__ void fill_group(const FillArgs::Segment& s, int64_t g) {
  constexpr int64_t W = sizeof(V) / 4;
  V* dst = reinterpret_cast<V*>(s.dst + g * s.dst_stride);
  const V* src = reinterpret_cast<const V*>(s.src + g * s.src_stride);
  const int64_t step = (int64_t)gridDim.x * kBlock, first = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  for (int64_t i = first; i < s.copy / W; i += step) dst[i] = src[i];
  for (int64_t i = s.zero_from / W + first; i < s.zero_to / W; i += step) dst[i] = V{};
}

__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// A launch takes the GPU about 2 us and the host 3.4 us whatever it does, so the diagonals of a new cache ride along: a prompt of
// 10 007 positions compressed into one, 81.6 -> 74.1 us against a launch of their own.
__global__ __launch_bounds__(kBlock) void fill_rows_kernel(FillArgs a) {
  if (blockIdx.y == a.n_segments) {
    if (blockIdx.z) return;
    for (int64_t i = blockIdx.x * kBlock + threadIdx.x; i < (int64_t)a.n_seeds * a.dim; i += gridDim.x * kBlock) {
      const int row = (int)(i / a.dim);
      uint64_t seed = a.seeds[0];                              // selects, not a dynamic index into kernel arguments
#pragma unroll
      for (int k = 1; k < TQ_SIGNS_MAX_SEEDS; ++k) seed = row == k ? a.seeds[k] : seed;
      a.signs[i] = (splitmix64(splitmix64(seed) + (uint64_t)(i - (int64_t)row * a.dim)) >> 63) ? 1.0f : -1.0f;
    }
    return;
  }
  const FillArgs::Segment& s = a.s[blockIdx.y];
  for (int64_t g = blockIdx.z; g < s.n_groups; g += gridDim.z) {
    if (s.wide) fill_group<uint4>(s, g);
    else fill_group<uint32_t>(s, g);
  }
}

int setup_rows(const char* who, const tq_fill_segment* segments, int n_segments, const uint64_t* seeds, int n_seeds, int dim,
               float* signs, hipStream_t stream) {
  if (n_segments < 0 || n_segments > TQ_FILL_MAX_SEGMENTS) return tq::fail(TQ_ERR_ARG, "%s: %d segments", who, n_segments);
  if (n_seeds < 0 || n_seeds > TQ_SIGNS_MAX_SEEDS) return tq::fail(TQ_ERR_ARG, "%s: %d seeds", who, n_seeds);
  if (n_seeds > 0 && dim < 1) return tq::fail(TQ_ERR_DIM, "%s: dim %d", who, dim);
  if ((n_segments > 0 && !segments) || (n_seeds > 0 && (!seeds || !signs))) return tq::fail(TQ_ERR_NULL, "%s: null pointer", who);
  if (n_seeds > 0 && !tq::aligned(signs, 4)) return tq::fail(TQ_ERR_ALIGN, "%s: misaligned pointer", who);
  FillArgs a{};
  a.n_segments = n_segments;
  a.n_seeds = n_seeds;
  a.dim = dim;
  a.signs = signs;
  for (int i = 0; i < n_seeds; ++i) a.seeds[i] = seeds[i];
  int64_t most = 0, groups = 1;
  for (int i = 0; i < n_segments; ++i) {
    const tq_fill_segment& g = segments[i];
    if (g.n_groups < 0 || g.copy_bytes < 0 || g.zero_from < 0 || g.zero_to < g.zero_from)
      return tq::fail(TQ_ERR_ARG, "%s: segment %d has a negative size", who, i);
    if (!g.dst || (g.copy_bytes > 0 && !g.src)) return tq::fail(TQ_ERR_NULL, "%s: null pointer", who);
    const int64_t bits = g.dst_group_stride | g.src_group_stride | g.copy_bytes | g.zero_from | g.zero_to |
                         (int64_t)(uintptr_t)g.dst | (int64_t)(uintptr_t)g.src;
    if (bits & 3) return tq::fail(TQ_ERR_ALIGN, "%s: segment %d is not made of 4-byte words", who, i);
    a.s[i] = {(uint32_t*)g.dst, (const uint32_t*)g.src, g.dst_group_stride / 4, g.src_group_stride / 4, g.copy_bytes / 4,
              g.zero_from / 4, g.zero_to / 4, g.n_groups, (bits & 15) == 0};
    const int64_t words = (g.copy_bytes + g.zero_to - g.zero_from) / 4 / ((bits & 15) == 0 ? 4 : 1);
    most = words > most ? words : most;
    groups = g.n_groups > groups ? g.n_groups : groups;
  }
  if (most == 0 && n_seeds == 0) return TQ_OK;
  const int64_t x = (std::max<int64_t>(most, (int64_t)n_seeds * dim) + kBlock - 1) / kBlock;
  const dim3 grid((unsigned)(x < 256 ? x : 256), n_segments + (n_seeds > 0 ? 1 : 0), (unsigned)(groups < 1024 ? groups : 1024));
  fill_rows_kernel<<<grid, kBlock, 0, stream>>>(a);
  TQ_CHECK_LAUNCH(who);
  return TQ_OK;
}
}  // namespace

extern "C" int tq_fill_rows(const tq_fill_segment* segments, int n_segments, tq_stream_t stream_) {
  return setup_rows("tq_fill_rows", segments, n_segments, nullptr, 0, 0, nullptr, (hipStream_t)stream_);
}

extern "C" int tq_random_signs(const uint64_t* seeds, int n_seeds, int dim, float* signs, tq_stream_t stream_) {
  if (dim < 1) return tq::fail(TQ_ERR_DIM, "tq_random_signs: dim %d", dim);
  return setup_rows("tq_random_signs", nullptr, 0, seeds, n_seeds, dim, signs, (hipStream_t)stream_);
}

extern "C" int tq_setup_rows(const tq_fill_segment* segments, int n_segments, const uint64_t* seeds, int n_seeds, int dim,
                             float* signs, tq_stream_t stream_) {
  return setup_rows("tq_setup_rows", segments, n_segments, seeds, n_seeds, dim, signs, (hipStream_t)stream_);
}

extern "C" int tq_prerotate_query(const void* q, int q_dtype, const float* signs, float* q_rot,
                                  int64_t n_heads, int dim, tq_stream_t stream_) {
  if (!tq::is_pow2(dim)) return tq::fail(TQ_ERR_DIM, "dim must be a power of 2, got %d", dim);
  if (dim < 32 || dim > 256) return tq::fail(TQ_ERR_DIM, "dim %d outside the supported range 32..256", dim);
  if (tq::check_dtype(q_dtype)) return tq::fail(TQ_ERR_DTYPE, "tq_prerotate_query: unknown q_dtype %d", q_dtype);
  if (n_heads < 0) return tq::fail(TQ_ERR_ARG, "tq_prerotate_query: negative n_heads");
  if (n_heads == 0) return TQ_OK;
  if (!q || !signs || !q_rot) return tq::fail(TQ_ERR_NULL, "tq_prerotate_query: null pointer");
  hipStream_t stream = (hipStream_t)stream_;
  const int grid = (int)((n_heads + kWavesPerBlock - 1) / kWavesPerBlock);
#define LAUNCH_PRE(T) \
  TQ_DISPATCH_DIM(dim, (prerotate_kernel<D_, T><<<grid, kBlock, 0, stream>>>((const T*)q, signs, q_rot, n_heads)))
  if (q_dtype == TQ_F32) { LAUNCH_PRE(float); }
  else if (q_dtype == TQ_F16) { LAUNCH_PRE(__half); }
  else { LAUNCH_PRE(__hip_bfloat16); }
#undef LAUNCH_PRE
  TQ_CHECK_LAUNCH("tq_prerotate_query launch");
  return TQ_OK;
}

extern "C" int tq_packed_qk_scores(const float* query, const uint32_t* k_packed, const float* k_norms,
                                   const float* centroids, const float* signs, float* scores, int n_heads,
                                   int64_t seq_len, int64_t packed_head_stride, int64_t norms_head_stride,
                                   int dim, int bits, tq_stream_t stream_) {
  if (int rc = tq::check_dim_bits(dim, bits)) return rc;
  if (n_heads < 0 || seq_len < 0) return tq::fail(TQ_ERR_ARG, "tq_packed_qk_scores: negative size");
  if (n_heads == 0 || seq_len == 0) return TQ_OK;
  if (!query || !k_packed || !k_norms || !centroids || !signs || !scores)
    return tq::fail(TQ_ERR_NULL, "tq_packed_qk_scores: null pointer");
  Codebook cb;
  for (int i = 0; i < 16; ++i) cb.c[i] = i < (1 << bits) ? centroids[i] : 0.0f;
  const float s = (float)(1.0 / sqrt((double)dim));
  hipStream_t stream = (hipStream_t)stream_;
  dim3 grid(grid_for_rows(seq_len), n_heads);
  TQ_DISPATCH_DIM(dim, TQ_DISPATCH_BITS(bits, (packed_qk_kernel<D_, B_><<<grid, kBlock, 0, stream>>>(
                                                  query, k_packed, k_norms, cb, signs, s, scores, seq_len,
                                                  packed_head_stride, norms_head_stride))));
  TQ_CHECK_LAUNCH("tq_packed_qk_scores launch");
  return TQ_OK;
}
