// Static quantise-dequantise of activations on the device: x -> bf16 bits of
// dec(static_encode(x / s)), without the codes in between.
#pragma once

#include "quant_device.h"

namespace hif8 {

typedef uint32_t qdq_u32x4 __attribute__((ext_vector_type(4)));

// Quantise-dequantise table of the kernels that encode and decode an
// activation in one go: entry i (the 13-bit sign / exponent / top-four-mantissa index of an FP32
// quotient x / s, the index of Tables::static_encode) holds the bf16 bits of
// dec(static_encode[i]).  One lookup instead of the encode and decode lookups;
// 16 KiB, copied into LDS by each block.
struct QdqTable {
  uint16_t v[8192];
};

constexpr QdqTable make_qdq_table() {
  QdqTable t{};
  for (uint32_t i = 0; i < 8192; ++i) t.v[i] = uint16_t(decode_bits(static_encode_bits(i << 19)) >> 16);
  return t;
}

static __device__ const QdqTable kQdqTable = make_qdq_table();

// Static encode + decode of 16 fp16/bf16 values into bf16 pairs through the
// quantise-dequantise table: the same reciprocal multiply, boundary test and
// IEEE-division redo as fast_encode_decode16, so each value equals
// dec(the standalone quant's code).  All 16 take the multiply first; one
// branch (rarely taken: a quotient within 8 ulps of an index boundary, or
// NaN) redoes the 16 with the division, so the kernel holds one copy of the
// division code per 16 values instead of one per pair.
template <bool kBf16>
__device__ __forceinline__ void fast_qdq16(const qdq_u32x4 a, const qdq_u32x4 b, float s, float r, const uint16_t *qdq,
                                           uint32_t (&p)[8]) {
  uint32_t u[16];
  bool redo = false;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t w = i < 4 ? a[i] : b[i - 4];
    const float q0 = lo_to_float<kBf16>(w) * r, q1 = hi_to_float<kBf16>(w) * r;
    redo |= near_index_boundary(q0) | near_index_boundary(q1);
    u[2 * i] = __float_as_uint(q0);
    u[2 * i + 1] = __float_as_uint(q1);
  }
  if (__builtin_expect(redo, 0)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t w = i < 4 ? a[i] : b[i - 4];
      const float q0 = lo_to_float<kBf16>(w) / s, q1 = hi_to_float<kBf16>(w) / s;
      // NaN quotients index the NaN entries of exponent 0xFF.
      u[2 * i] = __builtin_isnan(q0) ? 0x7FC00000u : __float_as_uint(q0);
      u[2 * i + 1] = __builtin_isnan(q1) ? 0x7FC00000u : __float_as_uint(q1);
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) p[i] = uint32_t(qdq[u[2 * i] >> 19]) | (uint32_t(qdq[u[2 * i + 1] >> 19]) << 16);
}

}  // namespace hif8
