// Gated delta rule over many tokens (linear-attention prefill) for gfx950, FP32.
//
// Per request and value head, over tokens t with decay g_t and strength beta_t:
//   S <- e^g S;  S <- S + k (beta (v - S^T k))^T;  o = S^T q        S [dk, dv]
// in chunks of 64 tokens (WY form).  With G the running sum of g in a chunk,
// L = strictly lower part of (beta_i k_i . k_j) e^(G_i - G_j):
//   U = (I + L)^-1 (beta v)         W = (I + L)^-1 (beta e^G k)
//   V' = U - W S                    o = (e^G q) S + tril(q k^T e^(G_i - G_j)) V'
//   S <- e^(G_last) S + (e^(G_last - G) k)^T V'
// Two launches:
//   * delta_chunk_kernel, one block per (request, head, chunk): everything that
//     does not depend on S.  I + L is solved by 16-row blocks: the 16 x 16
//     diagonal blocks are inverted by substitution, one per wavefront, and the
//     rest are matrix products over the columns [v | k], 64 per wavefront;
//   * delta_scan_kernel, one block per (request, head, 16 columns of dv): walks
//     the chunks with its [dk, 16] slice of S on chip.  Columns of S do not
//     interact, so the chain over chunks is the only serial one, and 32 heads
//     of dv = 128 give 256 blocks.
// Every product runs on v_mfma_f32_16x16x4_f32 (FP32 operands and sums).  Lane l
// holds A[l % 16][l / 16], B[l / 16][l % 16] and D[4 (l / 16) + e][l % 16], so
// four MFMAs over k = 4 (l / 16) + s (s = 0..3) take one float4 of a row-major A
// (or of a transposed B), and a D tile is the B operand of the next product as
// it stands.  The chunk kernel writes its results as such fragments (256
// floats each: one 1 KiB load); the scan reads the next chunk's while it works
// on the current one.
// The running sums G are FP64: an FP32 G of a few tens is off by 1e-6, and so
// then is every e^(G_i - G_j) of two neighbours.
// What bounds it (MI355X, 1000 tokens, 32 heads, dk = dv = 128; the torch form
// 2.7 ms in ~320 launches): the scan, 55.6 us, 3.5 us per chunk of which the
// 112 MFMAs of a wavefront, in chains of 32, are 1.5; the chunk kernel, 34.7
// us, writes 74 MB.
#include <math.h>

#include <algorithm>

#include "hif8_common.h"
#include "hif8_rocm.h"

namespace hif8 {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kC = 64;        // tokens per chunk
constexpr int kTiles = kC / 16;
constexpr int kThreads = 256;  // four wavefronts
constexpr int kFrag = 256;     // floats of one 16 x 16 fragment

struct DeltaShape {
  int heads, tokens, chunks, rep;              // rep: value heads per key head
  int64_t qb, qh, qt, kb, kh, kt, vb, vh, vt;  // element strides (batch, head, token); dims are contiguous
  int64_t gb, gh, gt, bb, bh, bt;              // of g and beta
  int64_t ob, oh, ot;                          // of the output
};

// Fragments of one (request, head, chunk), in floats from its first one.
template <int kDk>
struct ChunkLayout {
  static constexpr int kDkTiles = kDk / 16;
  static constexpr int kW = 0;                                  // [row tile][dk tile]: W
  static constexpr int kQ = kW + kTiles * kDkTiles * kFrag;     // [row tile][dk tile]: e^G q
  static constexpr int kK = kQ + kTiles * kDkTiles * kFrag;     // [dk tile][row tile]: (e^(G_last - G) k)^T
  static constexpr int kQK = kK + kTiles * kDkTiles * kFrag;    // [row tile][col tile], lower: q k^T decayed
  static constexpr int kDecay = kQK + kTiles * kTiles * kFrag;  // e^(G_last), padded to 64 floats
  static constexpr int kU = kDecay + 64;                        // [dv tile][row tile]: U
  static constexpr size_t floats(int dv) { return size_t(kU) + size_t(dv / 16) * kTiles * kFrag; }
};

__device__ __forceinline__ f32x4_t mfma(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// c + A B over 16 k, A and B as float4 per lane (k = 4 (l / 16) + s).
__device__ __forceinline__ f32x4_t mfma16(f32x4_t a, f32x4_t b, f32x4_t c) {
#pragma unroll
  for (int s = 0; s < 4; ++s) c = mfma(a[s], b[s], c);
  return c;
}
__device__ __forceinline__ f32x4_t ld4(const float *p) { return *reinterpret_cast<const f32x4_t *>(p); }
__device__ __forceinline__ void st4(float *p, f32x4_t v) { *reinterpret_cast<f32x4_t *>(p) = v; }

template <int kDk>
__global__ __launch_bounds__(kThreads, 2) void delta_chunk_kernel(
    const float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ v,
    const float *__restrict__ g, const float *__restrict__ beta, float *__restrict__ ws, const DeltaShape d, int dv) {
  using Layout = ChunkLayout<kDk>;
  constexpr int kPitch = kDk + 4, kLPitch = kC + 4, kDkTiles = kDk / 16;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float *ks = smem;               // k [token][dim], W in its place later
  float *lm = ks + kC * kPitch;   // L
  float *ti = lm + kC * kLPitch;  // inverses of the diagonal blocks of I + L: [block][16][20]
  double *gs = reinterpret_cast<double *>(ti + kTiles * 16 * 20);  // G
  float *bs = reinterpret_cast<float *>(gs + kC), *es = bs + kC;   // beta, e^G

  const int chunk = blockIdx.x % d.chunks, bh = blockIdx.x / d.chunks;
  const int b = bh / d.heads, h = bh - b * d.heads, hk = h / d.rep;
  const int t0 = chunk * kC, live = min(d.tokens - t0, kC);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
  const int fcol = lane & 15, fgrp = lane >> 4;
  const float *qp = q + b * d.qb + hk * d.qh + t0 * d.qt;
  const float *kp = k + b * d.kb + hk * d.kh + t0 * d.kt;
  const float *vp = v + b * d.vb + h * d.vh + t0 * d.vt;
  float *out = ws + size_t(blockIdx.x) * Layout::floats(dv);
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};

  // Tokens past the end are zero rows of no decay and no strength.
  constexpr int kLoads = kC * (kDk / 4) / kThreads;
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int e = tid + kThreads * i, r = e / (kDk / 4), c = e % (kDk / 4) * 4;
    st4(ks + r * kPitch + c, r < live ? ld4(kp + r * d.kt + c) : zero);
  }
  if (tid < kC) {
    const bool ok = tid < live;
    double sum = ok ? double(g[b * d.gb + h * d.gh + (t0 + tid) * d.gt]) : 0.;
    bs[tid] = ok ? beta[b * d.bb + h * d.bh + (t0 + tid) * d.bt] : 0.f;
#pragma unroll
    for (int o = 1; o < kC; o <<= 1) {
      const double left = __shfl_up(sum, o, kWave);
      if (lane >= o) sum += left;
    }
    gs[tid] = sum;
    es[tid] = expf(float(sum));
  }
  __syncthreads();

  // k k^T (wavefronts 0, 1) and q k^T (2, 3), lower tiles only: tile rows 3 and
  // 0, or 2 and 1, five tiles each.  Rows j of k are the A operand, so a lane
  // ends with four consecutive columns j of one row i.
  {
    const bool is_q = wave >= 2;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int it = wave & 1 ? 2 - half : 3 - 3 * half;
      const int i = 16 * it + fcol;
      f32x4_t br[kDkTiles];
#pragma unroll
      for (int c = 0; c < kDkTiles; ++c) {
        const int at = 16 * c + 4 * fgrp;
        if (is_q) br[c] = i < live ? ld4(qp + i * d.qt + at) : zero;
        else br[c] = ld4(ks + i * kPitch + at);
      }
      const double gi = gs[i];
      const float bi = bs[i];
      if (is_q) {
#pragma unroll
        for (int c = 0; c < kDkTiles; ++c)
          st4(out + Layout::kQ + (it * kDkTiles + c) * kFrag + 4 * lane, br[c] * es[i]);
      }
      for (int jt = 0; jt <= it; ++jt) {
        f32x4_t acc[2] = {zero, zero};
#pragma unroll
        for (int c = 0; c < kDkTiles; ++c)
          acc[c & 1] = mfma16(ld4(ks + (16 * jt + fcol) * kPitch + 16 * c + 4 * fgrp), br[c], acc[c & 1]);
        const f32x4_t sum = acc[0] + acc[1];
        f32x4_t o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = 16 * jt + 4 * fgrp + e;
          const float scale = expf(float(gi - gs[j])) * (is_q ? 1.f : bi);
          o[e] = (is_q ? j <= i : j < i) ? sum[e] * scale : 0.f;
        }
        if (is_q) st4(out + Layout::kQK + (it * kTiles + jt) * kFrag + 4 * lane, o);
        else st4(lm + i * kLPitch + 16 * jt + 4 * fgrp, o);
      }
    }
  }
  __syncthreads();

  // (I + L_ww)^-1 by forward substitution: lane j of the first 16 owns column j.
  {
    const float *lw = lm + 16 * wave * kLPitch + 16 * wave;
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float s = i == fcol ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) s -= lw[i * kLPitch + j] * x[j];
      x[i] = s;
    }
    if (lane < 16) {
#pragma unroll
      for (int i = 0; i < 16; ++i) ti[(16 * wave + i) * 20 + lane] = x[i];
    }
  }
  // k's fragments, transposed and scaled by e^(G_last - G).
  const double g_last = gs[kC - 1];
  for (int t = wave; t < kDkTiles; t += 4) {
#pragma unroll
    for (int c = 0; c < kTiles; ++c) {
      f32x4_t o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 16 * c + 4 * fgrp + e;
        o[e] = ks[i * kPitch + 16 * t + fcol] * expf(float(g_last - gs[i]));
      }
      st4(out + Layout::kK + (t * kTiles + c) * kFrag + 4 * lane, o);
    }
  }
  if (tid == 0) out[Layout::kDecay] = expf(float(g_last));
  __syncthreads();

  // (I + L) X = [beta v | beta e^G k], 16 columns at a time: X_I = T_I (R_I -
  // sum over J < I of L_IJ X_J).  A column tile of k is read and replaced by W by
  // one wavefront.
  const int dv_tiles = dv / 16, tiles = dv_tiles + kDkTiles;
  for (int n = wave; n < tiles; n += 4) {
    const bool is_v = n < dv_tiles;
    f32x4_t x[kTiles];
#pragma unroll
    for (int it = 0; it < kTiles; ++it) {
      f32x4_t r;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 16 * it + 4 * fgrp + e;
        const float y = is_v ? (i < live ? vp[i * d.vt + 16 * n + fcol] : 0.f)
                             : ks[i * kPitch + 16 * (n - dv_tiles) + fcol] * es[i];
        r[e] = bs[i] * y;
      }
      f32x4_t sub = zero;
#pragma unroll
      for (int jt = 0; jt < it; ++jt) sub = mfma16(ld4(lm + (16 * it + fcol) * kLPitch + 16 * jt + 4 * fgrp), x[jt], sub);
      x[it] = mfma16(ld4(ti + (16 * it + fcol) * 20 + 4 * fgrp), r - sub, zero);
      if (is_v) {
        st4(out + Layout::kU + (n * kTiles + it) * kFrag + 4 * lane, x[it]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) ks[(16 * it + 4 * fgrp + e) * kPitch + 16 * (n - dv_tiles) + fcol] = x[it][e];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < kDkTiles; ++c)
    st4(out + Layout::kW + (wave * kDkTiles + c) * kFrag + 4 * lane,
        ld4(ks + (16 * wave + fcol) * kPitch + 16 * c + 4 * fgrp));
}

// Block ids of one (request, head) are equal modulo 8: the column slices that
// read the same fragments share an XCD's L2.
template <int kDk>
__global__ __launch_bounds__(kThreads, 1) void delta_scan_kernel(const float *__restrict__ ws,
                                                                 float *__restrict__ state, float *__restrict__ o,
                                                                 const DeltaShape d, int dv, int groups) {
  using Layout = ChunkLayout<kDk>;
  constexpr int kDkTiles = kDk / 16, kOwn = kDkTiles / 4;  // S tiles per wavefront
  constexpr int kPitch = kDk + 4;
  __shared__ __attribute__((aligned(16))) float st[16 * kPitch];       // S^T: [column][dk]
  __shared__ __attribute__((aligned(16))) float vt[16 * (kC + 4)];     // V'^T: [column][token]
  const int slices = dv / 16;
  const int in_group = int(blockIdx.x) / 8;
  const int bh = int(blockIdx.x) % 8 + 8 * (in_group / slices), n = in_group % slices;
  if (bh >= groups) return;
  const int b = bh / d.heads, h = bh - b * d.heads;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
  const int fcol = lane & 15, fgrp = lane >> 4;
  const size_t per_chunk = Layout::floats(dv);
  const float *base = ws + size_t(bh) * d.chunks * per_chunk + 4 * lane;
  float *S = state + size_t(bh) * kDk * dv + 16 * n + fcol;
  float *op = o + b * d.ob + h * d.oh + 16 * n + fcol;

  struct Chunk {
    f32x4_t w[kDkTiles], q[kDkTiles], qk[kTiles], k[kOwn][kTiles], u;
    float decay;
  };
  auto load = [&](Chunk &c, int i) {
    const float *p = base + size_t(i) * per_chunk;
#pragma unroll
    for (int t = 0; t < kDkTiles; ++t) {
      c.w[t] = ld4(p + Layout::kW + (wave * kDkTiles + t) * kFrag);
      c.q[t] = ld4(p + Layout::kQ + (wave * kDkTiles + t) * kFrag);
    }
    c.u = ld4(p + Layout::kU + (n * kTiles + wave) * kFrag);
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
      c.qk[t] = ld4(p + Layout::kQK + (wave * kTiles + min(t, wave)) * kFrag);
#pragma unroll
    for (int s = 0; s < kOwn; ++s)
#pragma unroll
      for (int t = 0; t < kTiles; ++t) c.k[s][t] = ld4(p + Layout::kK + ((wave * kOwn + s) * kTiles + t) * kFrag);
    c.decay = p[Layout::kDecay - 4 * lane];
  };

  // This wavefront's tiles of S: rows 16 (wave kOwn + s) + 4 fgrp + e.
  f32x4_t own[kOwn];
#pragma unroll
  for (int s = 0; s < kOwn; ++s) {
    const int r = 16 * (wave * kOwn + s) + 4 * fgrp;
#pragma unroll
    for (int e = 0; e < 4; ++e) own[s][e] = S[size_t(r + e) * dv];
    st4(st + fcol * kPitch + r, own[s]);
  }
  __syncthreads();

  auto step = [&](const Chunk &c, int i) {
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t aw[2] = {zero, zero}, ao[2] = {zero, zero};
#pragma unroll
    for (int t = 0; t < kDkTiles; ++t) {
      const f32x4_t s = ld4(st + fcol * kPitch + 16 * t + 4 * fgrp);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        aw[t & 1] = mfma(c.w[t][e], s[e], aw[t & 1]);
        ao[t & 1] = mfma(c.q[t][e], s[e], ao[t & 1]);
      }
    }
    st4(vt + fcol * (kC + 4) + 16 * wave + 4 * fgrp, c.u - (aw[0] + aw[1]));
    lds_barrier();  // V' complete; every wavefront has read S
    f32x4_t vf[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) vf[t] = ld4(vt + fcol * (kC + 4) + 16 * t + 4 * fgrp);
#pragma unroll
    for (int s = 0; s < kOwn; ++s) own[s] *= c.decay;
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int s = 0; s < kOwn; ++s) own[s] = mfma(c.k[s][t][e], vf[t][e], own[s]);
#pragma unroll
    for (int s = 0; s < kOwn; ++s) st4(st + fcol * kPitch + 16 * (wave * kOwn + s) + 4 * fgrp, own[s]);
    f32x4_t out = ao[0] + ao[1];
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
      if (t <= wave) out = mfma16(c.qk[t], vf[t], out);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = i * kC + 16 * wave + 4 * fgrp + e;
      if (t < d.tokens) op[t * d.ot] = out[e];
    }
    lds_barrier();  // S complete; every wavefront has read V'
  };

  // Two chunks in registers, the next one loaded while a chunk is worked on
  // (the last one again past the end).
  Chunk c0, c1;
  load(c0, 0);
  for (int i = 0; i < d.chunks; i += 2) {
    load(c1, min(i + 1, d.chunks - 1));
    step(c0, i);
    if (i + 1 >= d.chunks) break;
    load(c0, min(i + 2, d.chunks - 1));
    step(c1, i + 1);
  }
#pragma unroll
  for (int s = 0; s < kOwn; ++s)
#pragma unroll
    for (int e = 0; e < 4; ++e) S[size_t(16 * (wave * kOwn + s) + 4 * fgrp + e) * dv] = own[s][e];
}

// ------------------------------------------------- around the delta rule

constexpr int kConvTokens = 16;  // tokens per thread

// Causal depthwise conv over time with the carried state, then SiLU, FP32: two
// channels and kConvTokens tokens per thread, so that a wavefront reads 256
// contiguous bytes of each token and every input once (plus kKw - 1 per run).
// Products and sums are rounded one by one, as elementwise FP32 operations are.
// The threads of the first tokens read the old state and write the new one.
// HBM-bound: 512 tokens of 8192 channels are 25 MB (MI355X 8.8 us; the
// elementwise operations it replaces took ~130).
template <int kKw>
__global__ __launch_bounds__(256) void conv_tokens_kernel(const uint16_t *__restrict__ x, int64_t ld, int channels,
                                                          const uint16_t *__restrict__ w, uint16_t *state,
                                                          float *__restrict__ out, int tokens) {
#pragma clang fp contract(off)
  const int c = 2 * (blockIdx.x * 256 + threadIdx.x), t0 = blockIdx.y * kConvTokens, b = blockIdx.z;
  if (c >= channels) return;
  auto bf = [](uint32_t h) { return __uint_as_float(h << 16); };
  const uint16_t *xr = x + size_t(b) * tokens * ld + c;
  uint16_t *st = state + (size_t(b) * channels + c) * (kKw - 1);
  auto input = [&](int t) { return *reinterpret_cast<const uint32_t *>(xr + size_t(t) * ld); };
  float w0[kKw], w1[kKw];
#pragma unroll
  for (int j = 0; j < kKw; ++j) {
    w0[j] = bf(w[size_t(c) * kKw + j]);
    w1[j] = bf(w[size_t(c + 1) * kKw + j]);
  }
  uint32_t win[kKw];  // inputs t - kKw + 1 .. t, channel c low
#pragma unroll
  for (int j = 0; j < kKw - 1; ++j)
    win[j] = t0 ? input(t0 - (kKw - 1) + j) : uint32_t(st[j]) | (uint32_t(st[kKw - 1 + j]) << 16);
  if (t0 == 0) {
    uint32_t next[kKw - 1];
#pragma unroll
    for (int j = 0; j < kKw - 1; ++j) {
      const int t = tokens + j - (kKw - 1);  // the last kKw - 1 of state and inputs
      next[j] = t >= 0 ? input(t) : uint32_t(st[tokens + j]) | (uint32_t(st[kKw - 1 + tokens + j]) << 16);
    }
#pragma unroll
    for (int j = 0; j < kKw - 1; ++j) {
      st[j] = uint16_t(next[j]);
      st[kKw - 1 + j] = uint16_t(next[j] >> 16);
    }
  }
  const int end = min(t0 + kConvTokens, tokens);
  float *o = out + (size_t(b) * tokens + t0) * channels + c;
  for (int t = t0; t < end; ++t, o += channels) {
    win[kKw - 1] = input(t);
    float a0 = bf(win[0] & 0xFFFFu) * w0[0], a1 = bf(win[0] >> 16) * w1[0];
#pragma unroll
    for (int j = 1; j < kKw; ++j) {
      a0 = a0 + bf(win[j] & 0xFFFFu) * w0[j];
      a1 = a1 + bf(win[j] >> 16) * w1[j];
    }
    *reinterpret_cast<float2 *>(o) = make_float2(a0 / (1.f + expf(-a0)), a1 / (1.f + expf(-a1)));
#pragma unroll
    for (int j = 0; j + 1 < kKw; ++j) win[j] = win[j + 1];
  }
}

// out[b, t, h] = bf16(o * rsqrt(mean(o^2) + eps) * w * silu(z)), one wavefront
// per (token, head) row of dv FP32 values (dv <= 256, even), two per lane and pass.
__global__ __launch_bounds__(256) void gated_norm_kernel(const float *__restrict__ o, int64_t ob, int64_t ot,
                                                         int64_t oh, const uint16_t *__restrict__ z, int64_t z_ld,
                                                         const uint16_t *__restrict__ w, uint16_t *__restrict__ out,
                                                         int tokens, int heads, int dv, int64_t first, int64_t rows,
                                                         float eps) {
  const int64_t row = first + int64_t(blockIdx.x) * 4 + threadIdx.x / kWave;  // (b, t, h)
  if (row >= rows) return;
  const int lane = threadIdx.x % kWave;
  const int64_t bt = row / heads;
  const int h = int(row - bt * heads), b = int(bt / tokens), t = int(bt - int64_t(b) * tokens);
  const float *src = o + b * ob + t * ot + h * oh;
  const uint16_t *zr = z + bt * z_ld + h * dv;
  auto bf = [](uint32_t v) { return __uint_as_float(v << 16); };
  float2 v[2];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int j = 2 * (lane + kWave * i);
    v[i] = j < dv ? *reinterpret_cast<const float2 *>(src + j) : make_float2(0.f, 0.f);
    ss += v[i].x * v[i].x + v[i].y * v[i].y;
  }
  const float r = rsqrtf(wave_sum(ss) / float(dv) + eps);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int j = 2 * (lane + kWave * i);
    if (j >= dv) continue;
    const uint32_t zw = *reinterpret_cast<const uint32_t *>(zr + j), ww = *reinterpret_cast<const uint32_t *>(w + j);
    const float z0 = bf(zw & 0xFFFFu), z1 = bf(zw >> 16);
    const float y0 = v[i].x * r * bf(ww & 0xFFFFu) * (z0 / (1.f + expf(-z0)));
    const float y1 = v[i].y * r * bf(ww >> 16) * (z1 / (1.f + expf(-z1)));
    *reinterpret_cast<uint32_t *>(out + row * dv + j) =
        uint32_t(float_to_bf16_bits(y0)) | (uint32_t(float_to_bf16_bits(y1)) << 16);
  }
}

template <int kDk>
int launch_delta(const float *q, const float *k, const float *v, const float *g, const float *beta, float *state,
                 float *out, float *ws, const DeltaShape &d, int batch, int dv, hipStream_t stream) {
  constexpr size_t kSmem = (kC * (kDk + 4) + kC * (kC + 4) + kTiles * 16 * 20 + 4 * kC) * sizeof(float);
  if (const int st = reserve_dynamic_lds(reinterpret_cast<const void *>(&delta_chunk_kernel<kDk>), kSmem,
                                         "hif8_gated_delta"))
    return st;
  const int groups = batch * d.heads;
  delta_chunk_kernel<kDk><<<unsigned(groups) * unsigned(d.chunks), kThreads, kSmem, stream>>>(q, k, v, g, beta, ws, d,
                                                                                              dv);
  if (const int st = check_launch("hif8_gated_delta (chunks)")) return st;
  delta_scan_kernel<kDk><<<unsigned((groups + 7) / 8 * 8) * unsigned(dv / 16), kThreads, 0, stream>>>(ws, state, out,
                                                                                                     d, dv, groups);
  return check_launch("hif8_gated_delta (scan)");
}

size_t delta_floats(int64_t dk, int64_t dv) {
  return dk == 64 ? ChunkLayout<64>::floats(int(dv)) : ChunkLayout<128>::floats(int(dv));
}

}  // namespace
}  // namespace hif8

using namespace hif8;

extern "C" size_t hif8_gated_delta_workspace_size(int64_t batch, int64_t heads, int64_t tokens, int64_t k_dim,
                                                  int64_t v_dim) {
  if (batch <= 0 || heads <= 0 || tokens <= 0 || (k_dim != 64 && k_dim != 128) || v_dim <= 0 || v_dim % 16 ||
      v_dim > 256)
    return 0;
  return size_t(batch) * size_t(heads) * size_t((tokens + kC - 1) / kC) * delta_floats(k_dim, v_dim) * sizeof(float);
}

extern "C" int hif8_gated_delta(const float *q, const float *k, const float *v, const float *g, const float *beta,
                                const int64_t *strides, float *state, float *out, int64_t batch, int64_t heads,
                                int64_t k_heads, int64_t tokens, int64_t k_dim, int64_t v_dim, void *workspace,
                                size_t workspace_bytes, hif8_stream_t stream) {
  clear_error();
  if (!q || !k || !v || !g || !beta || !strides || !state || !out || !workspace)
    return fail(HIF8_ERR_INVALID_ARGUMENT, "hif8_gated_delta: null pointer argument");
  if (batch <= 0 || heads <= 0 || k_heads <= 0 || heads % k_heads || tokens <= 0 || tokens > 0x7FFFFF00ll)
    return fail(HIF8_ERR_INVALID_ARGUMENT, "hif8_gated_delta: invalid dimensions");
  if ((k_dim != 64 && k_dim != 128) || v_dim <= 0 || v_dim % 16 || v_dim > 256)
    return fail(HIF8_ERR_UNSUPPORTED, "hif8_gated_delta: needs k_dim 64 or 128 and v_dim a multiple of 16 up to 256");
  const int64_t chunks = (tokens + kC - 1) / kC, slices = v_dim / 16;
  if (batch * heads > 0x7FFFFFF0ll / std::max<int64_t>(chunks, slices))
    return fail(HIF8_ERR_UNSUPPORTED, "hif8_gated_delta: too many chunks");
  DeltaShape d;
  d.heads = int(heads);
  d.tokens = int(tokens);
  d.chunks = int(chunks);
  d.rep = int(heads / k_heads);
  int64_t *const fields[18] = {&d.qb, &d.qh, &d.qt, &d.kb, &d.kh, &d.kt, &d.vb, &d.vh, &d.vt,
                               &d.gb, &d.gh, &d.gt, &d.bb, &d.bh, &d.bt, &d.ob, &d.oh, &d.ot};
  for (int i = 0; i < 18; ++i) *fields[i] = strides[i];
  for (int i = 0; i < 6; ++i)
    if (strides[i] % 4) return fail(HIF8_ERR_UNSUPPORTED, "hif8_gated_delta: q and k rows must be 16-byte aligned");
  if (!aligned(q, 16) || !aligned(k, 16))
    return fail(HIF8_ERR_UNSUPPORTED, "hif8_gated_delta: q and k rows must be 16-byte aligned");
  if (workspace_bytes < hif8_gated_delta_workspace_size(batch, heads, tokens, k_dim, v_dim) || !aligned(workspace, 256))
    return fail(HIF8_ERR_INVALID_ARGUMENT, "hif8_gated_delta: workspace too small or not 256-byte aligned");
  float *ws = static_cast<float *>(workspace);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (k_dim == 64) return launch_delta<64>(q, k, v, g, beta, state, out, ws, d, int(batch), int(v_dim), s);
  return launch_delta<128>(q, k, v, g, beta, state, out, ws, d, int(batch), int(v_dim), s);
}

extern "C" int hif8_conv_tokens(const uint16_t *x, int64_t ld, const uint16_t *conv_weight, uint16_t *conv_state,
                                float *out, int64_t batch, int64_t tokens, int64_t channels, int64_t conv_width,
                                hif8_stream_t stream) {
  clear_error();
  if (!x || !conv_weight || !conv_state || !out)
    return fail(HIF8_ERR_INVALID_ARGUMENT, "hif8_conv_tokens: null pointer argument");
  if (batch <= 0 || tokens <= 0 || channels <= 0 || ld < channels || tokens > 0x7FFFFF00ll ||
      channels > 0x7FFFFF00ll)
    return fail(HIF8_ERR_INVALID_ARGUMENT, "hif8_conv_tokens: invalid dimensions");
  const int64_t runs = (tokens + kConvTokens - 1) / kConvTokens;
  if (conv_width < 2 || conv_width > 4 || channels % 2 || ld % 2 || !aligned(x, 4) || !aligned(out, 8) ||
      batch > 65535 || runs > 65535)
    return fail(HIF8_ERR_UNSUPPORTED, "hif8_conv_tokens: needs 2 <= conv_width <= 4, even channels and row pitch, at "
                                      "most 65535 requests and %d tokens each", 65535 * kConvTokens);
  const dim3 grid(unsigned((channels / 2 + 255) / 256), unsigned(runs), unsigned(batch));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  auto go = [&](auto kern) {
    kern<<<grid, 256, 0, s>>>(x, ld, int(channels), conv_weight, conv_state, out, int(tokens));
  };
  if (conv_width == 2) go(conv_tokens_kernel<2>);
  else if (conv_width == 3) go(conv_tokens_kernel<3>);
  else go(conv_tokens_kernel<4>);
  return check_launch("hif8_conv_tokens");
}

extern "C" int hif8_gated_rms_norm(const float *o, int64_t o_batch, int64_t o_token, int64_t o_head,
                                   const uint16_t *z, int64_t z_ld, const uint16_t *weight, uint16_t *out,
                                   int64_t batch, int64_t tokens, int64_t heads, int64_t v_dim, float eps,
                                   hif8_stream_t stream) {
  clear_error();
  if (!o || !z || !weight || !out) return fail(HIF8_ERR_INVALID_ARGUMENT, "hif8_gated_rms_norm: null pointer argument");
  if (batch <= 0 || tokens <= 0 || heads <= 0 || v_dim <= 0 || tokens > 0x7FFFFFFFll || heads > 0x7FFFFFFFll ||
      z_ld < heads * v_dim)
    return fail(HIF8_ERR_INVALID_ARGUMENT, "hif8_gated_rms_norm: invalid dimensions");
  const int64_t rows = batch * tokens * heads;
  if (v_dim > 256 || v_dim % 2 || z_ld % 2 || o_batch % 2 || o_token % 2 || o_head % 2 || !aligned(o, 8) ||
      !aligned(z, 4) || !aligned(weight, 4) || !aligned(out, 4))
    return fail(HIF8_ERR_UNSUPPORTED, "hif8_gated_rms_norm: needs even v_dim <= 256, even strides and aligned rows");
  // A launch holds fewer than 2^32 threads.
  constexpr int64_t kStep = int64_t(1) << 24;
  for (int64_t first = 0; first < rows; first += kStep) {
    gated_norm_kernel<<<unsigned((std::min(kStep, rows - first) + 3) / 4), 256, 0,
                        reinterpret_cast<hipStream_t>(stream)>>>(o, o_batch, o_token, o_head, z, z_ld, weight, out,
                                                                 int(tokens), int(heads), int(v_dim), first, rows, eps);
    if (const int st = check_launch("hif8_gated_rms_norm")) return st;
  }
  return HIF8_OK;
}
