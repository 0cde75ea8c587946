// Where the bf16 activation of gemm_skinny_kernel sits in its fragments: plain
// C++, shared by the kernels that write and read them.
#pragma once

#include <cstddef>
#include <cstdint>

namespace hif8 {

constexpr int kStepK = 64;  // k per step: two fragments of 16 rows x 32 k

// 16-byte words before the piece of lane `lane` in half `half` of step `step` of
// row tile `tile` (steps per row tile: k padded to whole steps).  A row tile of K
// codes is 2 K words, so from K = 2^30 on this needs more than 32 bits.
constexpr size_t fragment_word(int64_t tile, int64_t steps, int64_t step, int half, int lane) {
  return ((size_t(tile) * size_t(steps) + size_t(step)) * 2 + size_t(half)) * 64 + size_t(lane);
}

}  // namespace hif8
