// Group-wise W4 helpers shared by the GEMV (w4g.hip) and the many-row product
// (w4m.hip).
#pragma once
#include "mm8t_common.h"

namespace rwkv7mi {

__device__ __forceinline__ f16x8 w4_nibbles_to_f16(uint32_t d) {
  // d = 8 nibbles n0..n7 (n_{2j} low nibble of byte j); out = [n0,n4,n1,n5,n2,n6,n3,n7] - 8.
  // fp16 pairs with exponent 0x64 hold 1024 + n (nibble in bits 0-3) or
  // 1024 + 16 n (bits 4-7): one packed add of -1032 or one packed fma by
  // 1/16 with -72 gives n - 8 exactly.  9 VALU ops per dword.
  const uint32_t d8 = d >> 8;
  const f16x2 a = __builtin_bit_cast(f16x2, and_or(d, 0x000F000Fu, 0x64006400u));
  const f16x2 b = __builtin_bit_cast(f16x2, and_or(d, 0x00F000F0u, 0x64006400u));
  const f16x2 c = __builtin_bit_cast(f16x2, and_or(d8, 0x000F000Fu, 0x64006400u));
  const f16x2 e = __builtin_bit_cast(f16x2, and_or(d8, 0x00F000F0u, 0x64006400u));
  const f16x2 off = {(_Float16)-1032.0f, (_Float16)-1032.0f};
  const f16x2 sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
  const f16x2 off16 = {(_Float16)-72.0f, (_Float16)-72.0f};
  const f16x2 p0 = a + off, p2 = c + off;
  const f16x2 p1 = __builtin_elementwise_fma(b, sixteenth, off16);
  const f16x2 p3 = __builtin_elementwise_fma(e, sixteenth, off16);
  return (f16x8){p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// Many-row product (w4m.hip), fp16 / bf16 activations: whether it takes these
// shapes, the workspace of its K splits (0: none), and its launches (a
// workspace below that runs unsplit).
bool w4m_supported(int64_t rows, int64_t O, int64_t I, int64_t group, int act_dtype);
int64_t w4m_workspace_bytes(int64_t rows, int64_t O, int64_t I, int act_dtype, bool aff);
int w4m_run(const void* x, const uint8_t* packed, const void* scales, const void* gbias, const void* bias,
            const void* residual, void* y, int64_t rows, int64_t O, int64_t I, int64_t group, int epilogue,
            int act_dtype, int scale_dtype, void* ws, int64_t ws_bytes, void* stream);

}  // namespace rwkv7mi
