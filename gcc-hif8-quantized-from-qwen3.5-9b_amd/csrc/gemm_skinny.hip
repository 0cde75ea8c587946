// GEMM of few activation rows, or of any K, for gfx950:
// C[m, n] = sum_k A[m, k] dec(W[n, k]) * ts[m] * cs[n] (+ b[n]), A already bf16.
//
// With up to ~64 rows the weight stream (N K bytes, read once) is what the
// call cannot do without, so the kernel is built like the GEMV: every wavefront
// streams its own weight codes from HBM straight into registers, decodes each
// one once (256-entry bf16 table in LDS, at address 0) into the A operand of
// v_mfma_f32_16x16x32_bf16 and multiplies it with all of the block's
// activation rows.  There is no LDS staging and no barrier in the K loop:
//   * a block owns kNT x 16 weight rows and kMT x 16 activation rows; its
//     kWaves wavefronts split K between them, 128 bytes (one cache line of a
//     weight row) at a time, and meet once in LDS at the end;
//   * lane l of a step of 64 k holds weight row l % 16, codes 16 (l / 16) ..
//     + 15: one 16-byte load per weight tile, decoded into the fragments of
//     two MFMAs.  The MFMA sums over k in any order as long as both operands
//     agree, so the activation fragment of step half h holds the 16-byte piece
//     A[l % 16][16 (l / 16) + 8 h ..].  The bf16 copy of the activation is laid
//     out in these fragments (1 KiB each, contiguous): in a row-major copy the
//     16 rows of a fragment sit K x 2 bytes apart, for the usual K on one L2
//     channel;
//   * kDepth steps of both operands are in flight per wavefront.
// What bounds it on MI355X: at M <= 32 over a wide weight the stream (24576 x
// 4096 at M = 16: 32.2 us with the decode launch, 3.6 TB/s; the 128 x 128 tiles,
// which decode W into LDS behind a barrier per step: 52 us); over narrow ones
// the two launches and the wavefront's chain of loads (2048 x 4096: 9.6 vs
// 22.5 us); from M = 48 on the fragment reads, M / 16 KiB per 64 x 16 codes
// through the vector cache (24576 x 4096: M = 64 44.6 us).  Read row-major the
// same fragments took 41.8 us at M = 32 instead of 36.5 and 61.6 at M = 64.
// The padding rows of the last fragment are not read: 4096 x 12288 at M = 5
// 22.6 -> 18.7 us, M = 24 26.6 -> 24.4.  Deeper pipelines (3, 4 steps), 16
// wavefronts, 64 weight rows per block (24576 x 4096 at M = 24: 38 us) and a
// start rotated per block measured the same or slower.
// K need not be a multiple of anything and weight rows need no alignment (the
// loads are emitted for byte alignment): the one partial step masks its codes
// to zero, and the bf16 copy is zero-padded to a multiple of 64.
#include <algorithm>

#include "fragment_layout.h"
#include "gemm_operand.h"

namespace hif8 {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_bytes __attribute__((aligned(1)));

// 16 codes -> 16 bf16 (lo = codes 0..7, hi = codes 8..15).
__device__ __forceinline__ void decode16(const uint16_t *lut, const u32x4 q, u32x4 &lo, u32x4 &hi) {
  uint32_t p[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = q[i];
    p[2 * i] = uint32_t(lut[w & 0xFFu]) | (uint32_t(lut[(w >> 8) & 0xFFu]) << 16);
    p[2 * i + 1] = uint32_t(lut[(w >> 16) & 0xFFu]) | (uint32_t(lut[w >> 24]) << 16);
  }
  lo = u32x4{p[0], p[1], p[2], p[3]};
  hi = u32x4{p[4], p[5], p[6], p[7]};
}

template <int kMT, int kNT, int kWaves, int kDepth>
__global__ __launch_bounds__(kWave * kWaves) void gemm_skinny_kernel(
    const uint16_t *__restrict__ A, int steps, const float *__restrict__ ts, const uint8_t *__restrict__ W,
    const float *__restrict__ cs, const void *__restrict__ bias, int bias_dtype, void *__restrict__ out,
    int out_dtype, int M, int N, int K, int n_tiles, int m_tiles, int n_first, int m_first) {
  constexpr int kBM = 16 * kMT, kBN = 16 * kNT;
  __shared__ __attribute__((aligned(16))) uint16_t lut[256];
  __shared__ __attribute__((aligned(16))) f32x4_t red[kWaves][kNT][kMT][kWave];

  // The row tiles (m_tiles of this launch, from m_first on) that read the same
  // weight rows are 8 block ids apart: one XCD, whose L2 then serves all but the
  // first.
  const int group = int(blockIdx.x) / (8 * m_tiles), in_group = int(blockIdx.x) - group * 8 * m_tiles;
  const int nt = n_first + group * 8 + (in_group & 7), mt = m_first + (in_group >> 3);
  if (nt >= n_tiles) return;
  const int n0 = nt * kBN, m0 = mt * kBM;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
  const int frow = lane & 15, fgrp = lane >> 4;

  for (int i = tid; i < 256; i += kWave * kWaves) lut[i] = uint16_t(decode_bits(uint32_t(i)) >> 16);

  // Rows past the end re-read the last one; their sums are not stored.  For the
  // activation this leaves the cache lines of a fragment's padding rows alone
  // (eight rows of a fragment are one line).
  const uint8_t *wrow[kNT];
  const u32x4 *afrag[kMT];
#pragma unroll
  for (int j = 0; j < kNT; ++j) wrow[j] = W + size_t(min(n0 + 16 * j + frow, N - 1)) * K + 16 * fgrp;
#pragma unroll
  for (int i = 0; i < kMT; ++i) {
    const int tile = min(m0 / 16 + i, (M - 1) / 16);
    afrag[i] = reinterpret_cast<const u32x4 *>(A) +
               fragment_word(tile, steps, 0, 0, 16 * fgrp + min(frow, M - 1 - 16 * tile));
  }

  struct Stage {
    u32x4 a[kMT][2], w[kNT];
  };
  // Step i of this wavefront: pairs of steps go round the wavefronts.
  auto step_k = [&](int i) { return ((i >> 1) * 2 * kWaves + 2 * wave + (i & 1)) * kStepK; };
  auto load = [&](Stage &s, int k0) {
#pragma unroll
    for (int t = 0; t < kMT; ++t) {
      const u32x4 *p = afrag[t] + fragment_word(0, 0, k0 / kStepK, 0, 0);
      s.a[t][0] = p[0];
      s.a[t][1] = p[kWave];
    }
#pragma unroll
    for (int j = 0; j < kNT; ++j) s.w[j] = *reinterpret_cast<const u32x4_bytes *>(wrow[j] + k0);
  };
  f32x4_t acc[kNT][kMT];
#pragma unroll
  for (int j = 0; j < kNT; ++j)
#pragma unroll
    for (int t = 0; t < kMT; ++t) acc[j][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto compute = [&](const Stage &s) {
#pragma unroll
    for (int j = 0; j < kNT; ++j) {
      u32x4 f[2];
      decode16(lut, s.w[j], f[0], f[1]);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < kMT; ++t)
          acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, f[h]),
                                                              __builtin_bit_cast(bf16x8_t, s.a[t][h]), acc[j][t], 0,
                                                              0, 0);
    }
  };

  // Full steps of this wavefront: those of whole pairs, then what the last,
  // incomplete round of pairs leaves it.
  const int full = K / kStepK, round = 2 * kWaves;
  const int mine = full / round * 2 + min(max(full % round - 2 * wave, 0), 2);
  // Loads without a branch around them, so that the compiler counts them and
  // each step waits for its own alone: a step past the last one re-reads it
  // (step 0 of the row where this wavefront has none).
  Stage st[kDepth];
  const auto safe_k = [&](int i) { return mine > 0 ? step_k(min(i, mine - 1)) : 0; };
  if (full > 0) {
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
      load(st[d], safe_k(d));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  lds_barrier();  // the table
  int i = 0;
  for (; i + kDepth < mine; i += kDepth) {
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
      compute(st[d]);
      __builtin_amdgcn_sched_barrier(0);  // the loads stay a whole round ahead of their use
      load(st[d], safe_k(i + kDepth + d));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int d = 0; d < kDepth; ++d)
    if (i + d < mine) compute(st[d]);
  // The partial step: codes past K become zero (the bf16 copy is zero there,
  // but a weight byte of the next row may be a NaN or Inf code).
  if (K % kStepK && (full >> 1) % kWaves == wave) {
    const int k0 = full * kStepK, left = K - k0 - 16 * fgrp;
    Stage s;
#pragma unroll
    for (int t = 0; t < kMT; ++t) {
      const u32x4 *p = afrag[t] + fragment_word(0, 0, k0 / kStepK, 0, 0);
      s.a[t][0] = p[0];
      s.a[t][1] = p[kWave];
    }
#pragma unroll
    for (int j = 0; j < kNT; ++j) {
      u32x4 q = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int b = 0; b < 16; ++b)
        if (b < left) q[b / 4] |= uint32_t(wrow[j][k0 + b]) << (8 * (b % 4));
      s.w[j] = q;
    }
    compute(s);
  }

  // The wavefronts' sums meet in LDS, added in wavefront order.  Lane l of a
  // 16 x 16 tile holds weight rows 4 (l / 16) .. + 3 of activation row l % 16.
#pragma unroll
  for (int j = 0; j < kNT; ++j)
#pragma unroll
    for (int t = 0; t < kMT; ++t) red[wave][j][t][lane] = acc[j][t];
  __syncthreads();
  constexpr int kTiles = kNT * kMT;
  const bool obf = out_dtype == HIF8_DTYPE_BF16;
  uint16_t *o = static_cast<uint16_t *>(out);
  const bool vec = N % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0;
  for (int tile = wave; tile < kTiles; tile += kWaves) {
    const int j = tile / kMT, t = tile % kMT;
    f32x4_t sum = red[0][j][t][lane];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) sum += red[w][j][t][lane];
    const int m = m0 + 16 * t + frow, n = n0 + 16 * j + 4 * fgrp;
    if (m >= M || n >= N) continue;
    const float s = ts[m];
    uint16_t h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = min(n + e, N - 1);
      float b = 0.f;
      if (bias) {
        const uint16_t hb = static_cast<const uint16_t *>(bias)[c];
        b = bias_dtype == HIF8_DTYPE_BF16 ? half_bits_to_float<true>(hb) : half_bits_to_float<false>(hb);
      }
      const float y = sum[e] * s * cs[c] + b;
      h[e] = obf ? float_to_bf16_bits(y) : float_to_f16_bits(y);
    }
    uint16_t *dst = o + size_t(m) * N + n;
    if (vec) {
      *reinterpret_cast<uint2 *>(dst) = make_uint2(uint32_t(h[0]) | (uint32_t(h[1]) << 16),
                                                   uint32_t(h[2]) | (uint32_t(h[3]) << 16));
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) dst[e] = h[e];
    }
  }
}

// Codes [rows, k] -> the bf16 fragments gemm_skinny_kernel reads: fragment
// (row tile, step, half) at 1 KiB each, rows padded to 16 and k to 64 with
// zeros.  One thread decodes the 16 codes that lane l holds of both halves;
// kVec: k % 16 == 0 and 16-byte aligned rows.
template <bool kVec>
__global__ __launch_bounds__(256) void decode_fragments_kernel(const uint8_t *__restrict__ a,
                                                               u32x4 *__restrict__ out, int rows, int k, int steps) {
  __shared__ __attribute__((aligned(16))) uint16_t lut[256];
  lut[threadIdx.x] = uint16_t(decode_bits(threadIdx.x) >> 16);
  lds_barrier();
  const int64_t total = int64_t((rows + 15) / 16) * steps * kWave;
  for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < total; i += int64_t(gridDim.x) * 256) {
    const int lane = int(i % kWave);
    const int64_t frag = i / kWave;  // row tile * steps + step
    const int row = int(frag / steps) * 16 + (lane & 15), c = int(frag % steps) * kStepK + 16 * (lane >> 4);
    const uint8_t *src = a + size_t(row) * k + c;
    u32x4 q = {0u, 0u, 0u, 0u};
    if (row < rows) {
      if constexpr (kVec) {
        if (c < k) q = *reinterpret_cast<const u32x4 *>(src);
      } else {
#pragma unroll
        for (int b = 0; b < 16; ++b)
          if (c + b < k) q[b / 4] |= uint32_t(src[b]) << (8 * (b % 4));
      }
    }
    u32x4 lo, hi;
    decode16(lut, q, lo, hi);
    out[fragment_word(0, 0, frag, 0, lane)] = lo;
    out[fragment_word(0, 0, frag, 1, lane)] = hi;
  }
}

template <int kMT, int kNT, int kWaves, int kDepth>
int launch_skinny_t(const LinearArgs &a, const uint16_t *act, int steps) {
  const int64_t n_tiles = (a.n + 16 * kNT - 1) / (16 * kNT), m_tiles = (a.m + 16 * kMT - 1) / (16 * kMT);
  // A launch holds fewer than 2^32 threads; more tiles go in several.
  constexpr int64_t kMaxBlocks = 0xFFFFFFFFll / (kWave * kWaves);
  const int64_t m_step = std::min(m_tiles, kMaxBlocks / 8), n_step = kMaxBlocks / (8 * m_step) * 8;
  for (int64_t nf = 0; nf < n_tiles; nf += n_step) {
    for (int64_t mf = 0; mf < m_tiles; mf += m_step) {
      const int64_t nb = (std::min(n_step, n_tiles - nf) + 7) / 8 * 8, mb = std::min(m_step, m_tiles - mf);
      gemm_skinny_kernel<kMT, kNT, kWaves, kDepth><<<unsigned(nb * mb), kWave * kWaves, 0, a.stream>>>(
          act, steps, a.act_scale, a.weight, a.channel_scale, a.bias, a.bias_dtype, a.out, a.out_dtype, int(a.m),
          int(a.n), int(a.k), int(n_tiles), int(mb), int(nf), int(mf));
      if (const int st = check_launch("soft_hif8 GEMM (few rows)")) return st;
    }
  }
  return HIF8_OK;
}

}  // namespace

size_t skinny_workspace_size(int64_t m, int64_t k) {
  return size_t((m + 15) / 16 * 16) * size_t((k + kStepK - 1) / kStepK * kStepK) * 2;
}

int launch_decode_fragments(const LinearArgs &a, uint16_t *act) {
  const int steps = int((a.k + kStepK - 1) / kStepK);
  const uint8_t *codes = static_cast<const uint8_t *>(a.act);
  const int64_t items = (a.m + 15) / 16 * steps * kWave;
  const unsigned blocks = unsigned(std::min<int64_t>((items + 255) / 256, 4096));
  u32x4 *out = reinterpret_cast<u32x4 *>(act);
  if (a.k % 16 == 0 && aligned(codes, 16))
    decode_fragments_kernel<true><<<blocks, 256, 0, a.stream>>>(codes, out, int(a.m), int(a.k), steps);
  else
    decode_fragments_kernel<false><<<blocks, 256, 0, a.stream>>>(codes, out, int(a.m), int(a.k), steps);
  return check_launch("soft_hif8 GEMM (activation decode)");
}

int launch_gemm_skinny(const LinearArgs &a, const uint16_t *act) {
  const int steps = int((a.k + kStepK - 1) / kStepK);
  // 32 weight rows per block share the activation fragments of a step (wide N,
  // or row tiles that fill the CUs); otherwise 16 give more CUs a block, and
  // eight wavefronts each a shorter chain.  MI355X, with the decode launch:
  // 24576 x 4096 at M = 24 34.2 us (16 rows per block: 39.8), M = 64 44.9 (58.5);
  // 2048 x 4096 at M = 24 10.6 (32 rows per block: 13.0), M = 64 14.5 (17.9).
  const bool wide = (a.n + 15) / 16 * ((a.m + 63) / 64) > 256;
  // Eight wavefronts in the wide blocks too while the sums of up to 32 rows leave
  // their meeting place small (8192 x 4096: M = 5 13.5 us, four wavefronts 14.9;
  // 24576 x 4096: M = 24 34.2 against 35.2, but M = 40 41.4 against 39.0).
  switch (std::min<int64_t>((a.m + 15) / 16, 4)) {
    case 1: return wide ? launch_skinny_t<1, 2, 8, 2>(a, act, steps) : launch_skinny_t<1, 1, 8, 2>(a, act, steps);
    case 2: return wide ? launch_skinny_t<2, 2, 8, 2>(a, act, steps) : launch_skinny_t<2, 1, 8, 2>(a, act, steps);
    case 3: return wide ? launch_skinny_t<3, 2, 4, 2>(a, act, steps) : launch_skinny_t<3, 1, 8, 2>(a, act, steps);
    default: return wide ? launch_skinny_t<4, 2, 4, 2>(a, act, steps) : launch_skinny_t<4, 1, 8, 2>(a, act, steps);
  }
}

}  // namespace hif8
