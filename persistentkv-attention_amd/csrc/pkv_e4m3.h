// pkv_e4m3.h — the OCP fp8 e4m3 encode of the KV append into fp8 pools (the bytes of
// torch's float8_e4m3fn cast), kept in one place for any kernel that stores fp8 K/V.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

namespace pkv {

// OCP e4m3 bytes of y0 (low byte) and y1: |y| clamped to 448, rounded to the nearest value
// with ties to the even code (v_cvt_pk_fp8_f32); NaN keeps its sign (0x7f / 0xff).  The
// conversion of two values is ~10 instructions, ~60 through the fp32 bits.
__device__ inline uint32_t e4m3_encode2(float y0, float y1) {
  const float c0 = fminf(fmaxf(y0, -448.0f), 448.0f), c1 = fminf(fmaxf(y1, -448.0f), 448.0f);
  uint32_t r = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c0, c1, 0, false) & 0xFFFFu;
  if (y0 != y0) r = (r & 0xFF00u) | 0x7Fu | ((__float_as_uint(y0) >> 24) & 0x80u);
  if (y1 != y1) r = (r & 0xFFu) | 0x7F00u | ((__float_as_uint(y1) >> 16) & 0x8000u);
  return r;
}

// Two 16-bit values (fp16, or bf16 when BF16_IN), low half first, to two e4m3 bytes of
// x / scale, low byte first.
template <bool BF16_IN>
__device__ inline float half_bits_to_float(uint32_t h) {
  if constexpr (BF16_IN) return __uint_as_float(h << 16);
  return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}
template <bool BF16_IN>
__device__ inline uint32_t e4m3_pack2(uint32_t x2, float scale) {
  return e4m3_encode2(half_bits_to_float<BF16_IN>(x2 & 0xFFFFu) / scale,
                      half_bits_to_float<BF16_IN>(x2 >> 16) / scale);
}

}  // namespace pkv
