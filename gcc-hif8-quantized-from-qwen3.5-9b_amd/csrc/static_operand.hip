// The GEMM's activation operand straight from fp16 / bf16 x: bf16 bits of
// dec(static_encode(x / s)) with one fixed scale, equal to hif8_static_quant
// followed by the decode of its codes.  One launch of 2 bytes in and 2 out per
// element replaces two (2 in, 1 out; 1 in, 2 out) and a launch gap: MI355X, 24
// x 4096 4.5 us instead of 4.3 + 3.4, a layer of 512 rows (K 4096 and 12288) 6.0
// instead of 5.2 + 4.9 on average, of 4096 rows 21 us (4.5 TB/s).
#include <algorithm>

#include "fragment_layout.h"
#include "gemm_operand.h"
#include "qdq_device.h"

namespace hif8 {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;

// kFrag: the fragment order of gemm_skinny_kernel, rows padded to 16 and k to
// 64 with zeros; otherwise row-major.  kVec: k % 16 == 0 and 16-byte aligned x
// (row-major takes nothing else).  One thread makes 16 consecutive elements of
// a row; the next item is loaded while one is converted.  The 16 KiB table is
// requested first, so its LDS stores wait for it alone.
template <bool kBf16, bool kFrag, bool kVec>
__global__ __launch_bounds__(kThreads) void static_operand_kernel(const uint16_t *__restrict__ x,
                                                                  const float *__restrict__ fixed,
                                                                  u32x4 *__restrict__ out,
                                                                  float *__restrict__ row_scale, int rows, int k,
                                                                  int steps, int64_t items) {
  static_assert(kFrag || kVec, "row-major output takes aligned rows");
  __shared__ __attribute__((aligned(16))) uint16_t qdq[8192];
  constexpr int kWords = 8192 * 2 / 16 / kThreads;
  u32x4 table[kWords];
#pragma unroll
  for (int i = 0; i < kWords; ++i)
    table[i] = reinterpret_cast<const u32x4 *>(kQdqTable.v)[threadIdx.x + i * kThreads];
  const int64_t stride = int64_t(gridDim.x) * kThreads;
  int64_t item = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  const u32x4 zero = {0u, 0u, 0u, 0u};
  u32x4 a = zero, b = zero;
  int left = 0;  // elements of the item that exist
  auto fetch = [&](int64_t it) {
    it = std::min(it, items - 1);
    if constexpr (!kFrag) {
      const u32x4 *src = reinterpret_cast<const u32x4 *>(x + it * 16);
      a = src[0];
      b = src[1];
      left = 16;
    } else {
      const int lane = int(it % kWave);
      const int64_t frag = it / kWave;
      const int row = int(frag / steps) * 16 + (lane & 15), c = int(frag % steps) * kStepK + 16 * (lane >> 4);
      left = row < rows ? k - c : 0;
      const uint16_t *src = x + size_t(std::min(row, rows - 1)) * k;
      if constexpr (kVec) {  // all or nothing
        const u32x4 *p = reinterpret_cast<const u32x4 *>(src + (c < k ? c : 0));
        a = p[0];
        b = p[1];
      } else {
        a = b = zero;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (e < left) a[e / 2] |= uint32_t(src[c + e]) << (16 * (e % 2));
          if (e + 8 < left) b[e / 2] |= uint32_t(src[c + e + 8]) << (16 * (e % 2));
        }
      }
    }
  };
  fetch(item);
  const float s = fixed[0];
  for (int64_t r = item; r < rows; r += stride) row_scale[r] = s;
#pragma unroll
  for (int i = 0; i < kWords; ++i) reinterpret_cast<u32x4 *>(qdq)[threadIdx.x + i * kThreads] = table[i];
  const float rcp = __builtin_amdgcn_rcpf(s);
  lds_barrier();
  for (; item < items; item += stride) {
    const u32x4 ca = a, cb = b;
    const int live = left;
    fetch(item + stride);
    uint32_t p[8];
    fast_qdq16<kBf16>(ca, cb, s, rcp, qdq, p);
    if constexpr (kFrag) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (live <= 2 * i) p[i] = 0u;
        else if (live == 2 * i + 1) p[i] &= 0xFFFFu;
      }
    }
    const u32x4 lo = {p[0], p[1], p[2], p[3]}, hi = {p[4], p[5], p[6], p[7]};
    if constexpr (kFrag) {
      out[fragment_word(0, 0, item / kWave, 0, int(item % kWave))] = lo;
      out[fragment_word(0, 0, item / kWave, 1, int(item % kWave))] = hi;
    } else {
      out[2 * item] = lo;
      out[2 * item + 1] = hi;
    }
  }
}

}  // namespace

int launch_static_operand(const void *x, bool bf16, const float *fixed, uint16_t *out, float *row_scale, int64_t rows,
                          int64_t k, bool fragments, hipStream_t stream) {
  const int64_t steps = (k + kStepK - 1) / kStepK;
  const int64_t items = fragments ? (rows + 15) / 16 * steps * kWave : rows * k / 16;
  const bool vec = k % 16 == 0 && aligned(x, 16);
  if (!fragments && !vec) return fail(HIF8_ERR_UNSUPPORTED, "hif8_static_linear: x must be 16-byte aligned");
  const unsigned blocks = unsigned(std::min<int64_t>((items + kThreads - 1) / kThreads, 256 * 16));
  const uint16_t *xs = static_cast<const uint16_t *>(x);
  auto go = [&](auto kern) {
    kern<<<blocks, kThreads, 0, stream>>>(xs, fixed, reinterpret_cast<u32x4 *>(out), row_scale, int(rows), int(k),
                                          int(steps), items);
  };
  if (!fragments) bf16 ? go(static_operand_kernel<true, false, true>) : go(static_operand_kernel<false, false, true>);
  else if (vec) bf16 ? go(static_operand_kernel<true, true, true>) : go(static_operand_kernel<false, true, true>);
  else bf16 ? go(static_operand_kernel<true, true, false>) : go(static_operand_kernel<false, true, false>);
  return check_launch("hif8_static_linear (activation)");
}

}  // namespace hif8
