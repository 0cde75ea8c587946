// The GEMM's bf16 activation operand: how it is made and which kernel reads it.
#pragma once

#include "linear.h"

namespace hif8 {

// bf16 bits of dec(static_encode(x / fixed[0])) of x [rows, k], row-major (k %
// 16 == 0, 16-byte aligned) or in the fragments of gemm_skinny_kernel (any k
// and alignment), and row_scale[r] = fixed[0] (static_operand.hip).
int launch_static_operand(const void *x, bool bf16, const float *fixed, uint16_t *out, float *row_scale, int64_t rows,
                          int64_t k, bool fragments, hipStream_t stream);

// gemm_skinny.hip.  Fragments of activation codes (a.act) in `act`
// (skinny_workspace_size(m, k) bytes, 256-byte aligned), and the GEMM over
// fragments already there.
size_t skinny_workspace_size(int64_t m, int64_t k);
int launch_decode_fragments(const LinearArgs &a, uint16_t *act);
int launch_gemm_skinny(const LinearArgs &a, const uint16_t *act);

// out = static_quant(x) W^T ...: a.act fp16 / bf16 x (a.act_kind kActF16 /
// kActBf16), a.act_scale the fixed scale, m > 4 or k % 16 != 0; a 256-byte
// aligned a.workspace of gemm_static_workspace_size(m, n, k) bytes (gemm.hip).
int launch_gemm_static(const LinearArgs &a);
size_t gemm_static_workspace_size(int64_t m, int64_t n, int64_t k);

}  // namespace hif8
