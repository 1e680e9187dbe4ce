// Packing of index rows into words and back, as operations of their own (packing.py:26-87).
//
// Both are bound by memory: 141 bytes per row of 128 indices and one packed row of 52 bytes at three bits.  As a chain of
// tensor operations in 64-bit integers (shift, mask, pad, sum) they moved 1 to 2 KB per index row: 100 003 rows of 128
// at three bits took 130 us (unpack) and 140 us (pack), of a PolarQuantizer round trip of 332 us, which took 42 us with these kernels (24 us since it goes without words).  Here a lane takes
// what one wide access holds: 16 indices of the output (one 16-byte store), or one packed word of the output (two to
// eight 4-byte loads).
#include "tq_common.h"

namespace {

using namespace tqd;

constexpr int kBlock = 256;

// sixteen fields of BITS bits as bytes
template <int BITS>
__device__ __forceinline__ uint4 spread16(uint64_t x) {
  uint32_t o[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    o[q] = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[q] |= ((uint32_t)(x >> (BITS * (4 * q + i))) & Pk<BITS>::MASK) << (8 * i);
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// Rows of a multiple of 16 indices, 16-byte aligned: lane t writes indices 16 t .. 16 t + 15 of the flat output.
// At three bits they lie in up to three words (ten fields each); every word that holds one of them is inside the row,
// the clamp keeps the loads of words that are not needed there as well.
template <int BITS>
__global__ __launch_bounds__(kBlock) void unpack16_kernel(const uint32_t* __restrict__ packed, uint4* __restrict__ out,
                                                          uint32_t n, uint32_t per_row, uint32_t pd) {
  const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= n) return;
  const uint32_t row = t / per_row, e0 = 16 * (t - row * per_row);
  const uint32_t* src = packed + (uint64_t)row * pd;
  const uint32_t w0 = e0 / Pk<BITS>::VPW, s = BITS * (e0 % Pk<BITS>::VPW);
  uint64_t x;
  if constexpr (BITS == 3) {
    const uint32_t last = pd - 1;
    const uint64_t a = src[w0] & 0x3FFFFFFFu, b = src[min(w0 + 1, last)] & 0x3FFFFFFFu, c = src[min(w0 + 2, last)];
    x = ((a | (b << 30)) >> s) | (c << (60 - s));
  } else if constexpr (BITS == 4) {
    x = (uint64_t)src[w0] | ((uint64_t)src[w0 + 1] << 32);
  } else {
    x = src[w0] >> s;
  }
  out[t] = spread16<BITS>(x);
}

// any row length and alignment: a lane writes one index
template <int BITS>
__global__ __launch_bounds__(kBlock) void unpack_kernel(const uint32_t* __restrict__ packed, uint8_t* __restrict__ out,
                                                        int64_t n, int32_t dim, int32_t pd) {
  for (int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x; t < n; t += (int64_t)gridDim.x * kBlock) {
    const int64_t row = t / dim;
    const int32_t e = (int32_t)(t - row * dim);
    out[t] = (uint8_t)((packed[row * pd + e / Pk<BITS>::VPW] >> (BITS * (e % Pk<BITS>::VPW))) & Pk<BITS>::MASK);
  }
}

// Lane t builds packed word t: the sum of its indices, each shifted to its field and none masked (an index past the
// width reaches into the fields above it, as the sum of the shifted integers does).  WIDE (bytes, rows of a multiple
// of four): 4-byte loads; at three bits a word's ten bytes start at a multiple of two.
template <int BITS, typename T, bool WIDE>
__global__ __launch_bounds__(kBlock) void pack_kernel(const T* __restrict__ idx, uint32_t* __restrict__ packed,
                                                      int64_t n, int32_t dim, int32_t pd) {
  constexpr int VPW = Pk<BITS>::VPW;
  for (int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x; t < n; t += (int64_t)gridDim.x * kBlock) {
    int64_t row;
    if (n < ((int64_t)1 << 32)) row = (uint32_t)t / (uint32_t)pd;
    else row = t / pd;
    const int32_t e0 = (int32_t)(t - row * pd) * VPW, have = min(VPW, dim - e0);
    uint32_t word = 0;
    if constexpr (WIDE) {
      constexpr int kLoads = BITS == 3 ? 3 : VPW / 4;
      const uint32_t* src = reinterpret_cast<const uint32_t*>(idx + row * dim);
      const int32_t d0 = e0 >> 2, last = (dim >> 2) - 1;
      uint32_t d[kLoads];
#pragma unroll
      for (int i = 0; i < kLoads; ++i) d[i] = src[min(d0 + i, last)];
      if constexpr (BITS == 3) {                                       // ten bytes from byte 0 or 2 of twelve
        const int sh = (e0 & 2) * 8;
        d[0] = (uint32_t)((((uint64_t)d[1] << 32) | d[0]) >> sh);
        d[1] = (uint32_t)((((uint64_t)d[2] << 32) | d[1]) >> sh);
        d[2] >>= sh;
      }
#pragma unroll
      for (int i = 0; i < VPW; ++i)
        if (i < have) word += ((d[i >> 2] >> (8 * (i & 3))) & 0xFFu) << (BITS * i);
    } else {
      const T* src = idx + row * dim + e0;
      for (int i = 0; i < have; ++i) word += (uint32_t)src[i] << (BITS * i);
    }
    packed[t] = word;
  }
}

int blocks_of(int64_t n) {
  const int64_t b = (n + kBlock - 1) / kBlock;
  return (int)(b < (1 << 20) ? b : (1 << 20));
}

}  // namespace

extern "C" int tq_unpack_indices(const uint32_t* packed, uint8_t* indices, int64_t n_rows, int words_per_row, int dim,
                                 int bits, tq_stream_t stream_) {
  const char* who = "tq_unpack_indices";
  const int vpw = tq::vals_per_word(bits);
  if (!vpw) return tq::fail(TQ_ERR_BITS, "Unsupported bit width: %d. Use 1-4.", bits);
  if (n_rows < 0 || words_per_row < 1 || dim < 1 || dim > (int64_t)words_per_row * vpw)
    return tq::fail(TQ_ERR_ARG, "%s: %lld rows of %d indices in %d words", who, (long long)n_rows, dim, words_per_row);
  if (n_rows == 0) return TQ_OK;
  if (!packed || !indices) return tq::fail(TQ_ERR_NULL, "%s: null pointer", who);
  if (!tq::aligned(packed, 4)) return tq::fail(TQ_ERR_ALIGN, "%s: misaligned pointer", who);
  hipStream_t stream = (hipStream_t)stream_;
  const int64_t n = n_rows * dim;
  if (dim % 16 == 0 && tq::aligned(indices, 16) && n / 16 < ((int64_t)1 << 31)) {
    const uint32_t n16 = (uint32_t)(n / 16);
    TQ_DISPATCH_BITS(bits, (unpack16_kernel<B_><<<(n16 + kBlock - 1) / kBlock, kBlock, 0, stream>>>(
                                packed, (uint4*)indices, n16, (uint32_t)dim / 16, (uint32_t)words_per_row)));
  } else {
    TQ_DISPATCH_BITS(bits, (unpack_kernel<B_><<<blocks_of(n), kBlock, 0, stream>>>(packed, indices, n, dim, words_per_row)));
  }
  TQ_CHECK_LAUNCH("tq_unpack_indices launch");
  return TQ_OK;
}

extern "C" int tq_pack_indices(const void* indices, int index_bytes, uint32_t* packed, int64_t n_rows, int dim, int bits,
                               tq_stream_t stream_) {
  const char* who = "tq_pack_indices";
  const int vpw = tq::vals_per_word(bits);
  if (!vpw) return tq::fail(TQ_ERR_BITS, "Unsupported bit width: %d. Use 1-4.", bits);
  if (index_bytes != 1 && index_bytes != 4 && index_bytes != 8)
    return tq::fail(TQ_ERR_DTYPE, "%s: indices of %d bytes", who, index_bytes);
  if (n_rows < 0 || dim < 1) return tq::fail(TQ_ERR_ARG, "%s: %lld rows of %d indices", who, (long long)n_rows, dim);
  if (n_rows == 0) return TQ_OK;
  if (!indices || !packed) return tq::fail(TQ_ERR_NULL, "%s: null pointer", who);
  if (!tq::aligned(indices, index_bytes) || !tq::aligned(packed, 4))
    return tq::fail(TQ_ERR_ALIGN, "%s: misaligned pointer", who);
  hipStream_t stream = (hipStream_t)stream_;
  const int pd = tq::packed_dim(dim, bits);
  const int64_t n = n_rows * pd;
  const int grid = blocks_of(n);
  if (index_bytes == 1 && dim % 4 == 0 && tq::aligned(indices, 4)) {
    TQ_DISPATCH_BITS(bits, (pack_kernel<B_, uint8_t, true><<<grid, kBlock, 0, stream>>>((const uint8_t*)indices, packed, n, dim, pd)));
  } else if (index_bytes == 1) {
    TQ_DISPATCH_BITS(bits, (pack_kernel<B_, uint8_t, false><<<grid, kBlock, 0, stream>>>((const uint8_t*)indices, packed, n, dim, pd)));
  } else if (index_bytes == 4) {
    TQ_DISPATCH_BITS(bits, (pack_kernel<B_, uint32_t, false><<<grid, kBlock, 0, stream>>>((const uint32_t*)indices, packed, n, dim, pd)));
  } else {
    TQ_DISPATCH_BITS(bits, (pack_kernel<B_, uint64_t, false><<<grid, kBlock, 0, stream>>>((const uint64_t*)indices, packed, n, dim, pd)));
  }
  TQ_CHECK_LAUNCH("tq_pack_indices launch");
  return TQ_OK;
}
