// Device helpers the attention kernels share: MFMA on 16-bit operands held as
// raw bits, packing and hi / lo splitting of fp32 values, and wave-wide
// column maxima.
#pragma once

#include "cab_internal.h"

namespace cab {

template <bool BF16>
__device__ __forceinline__ f32x4 mfma16(const u32x4& a, const u32x4& b, const f32x4& c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

template <bool BF16>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  if constexpr (BF16) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};  // v_cvt_pk_bf16_f32, RNE
    return __builtin_bit_cast(uint32_t, v);
  } else {
    return static_cast<uint32_t>(f32_to_f16(lo)) | (static_cast<uint32_t>(f32_to_f16(hi)) << 16);
  }
}

// fp32 -> bf16 pair split of two values: {hi, lo} with hi = bf16(x) and
// lo = bf16(x - hi), both round-to-nearest-even (x - hi is exact in fp32).
__device__ __forceinline__ u32x2 split2(float x0, float x1) {
  const uint32_t hi = pack2<true>(x0, x1);
  const float h0 = __builtin_bit_cast(float, hi << 16);
  const float h1 = __builtin_bit_cast(float, hi & 0xffff0000u);
  return u32x2{hi, pack2<true>(x0 - h0, x1 - h1)};
}

// Eight consecutive fp32 values (x0, x1) -> bf16x8 hi and lo operands.
__device__ __forceinline__ void split8(const f32x4& x0, const f32x4& x1, u32x4& hi, u32x4& lo) {
  const u32x2 a = split2(x0[0], x0[1]), b = split2(x0[2], x0[3]);
  const u32x2 e = split2(x1[0], x1[1]), f = split2(x1[2], x1[3]);
  hi = u32x4{a[0], b[0], e[0], f[0]};
  lo = u32x4{a[1], b[1], e[1], f[1]};
}

// gfx950 lane swaps between the two halves of two registers (v_permlane32_swap:
// 32-lane halves; v_permlane16_swap: odd and even 16-lane rows), written as
// inline asm because the compiler's builtins return the first result twice.
// The s_nop gives the two wait states a swap needs after a VALU write of
// its operands.
__device__ __forceinline__ void lane_swap32(uint32_t& a, uint32_t& b) {
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ void lane_swap16(uint32_t& a, uint32_t& b) {
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}

// Maxima over the four lane groups (lanes c + 16 g, g = 0..3) of two
// registers at once, without an LDS round trip. In: x0, x1 hold per-lane
// partial maxima of query column c = lane % 16 for query tiles 0 and 1.
// Out: each holds its tile's full column maximum in every lane.
__device__ __forceinline__ void colmax2(float& x0, float& x1) {
  uint32_t a = __builtin_bit_cast(uint32_t, x0), b = __builtin_bit_cast(uint32_t, x1);
  lane_swap32(a, b);  // one register holds both tiles' lower halves, the other the upper
  float y = __builtin_fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
  // y: tile 0 merged over g and g ^ 2 in one 32-lane half, tile 1 in the other.
  a = b = __builtin_bit_cast(uint32_t, y);
  lane_swap16(a, b);  // rows g and g ^ 1 side by side
  y = __builtin_fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
  a = b = __builtin_bit_cast(uint32_t, y);
  lane_swap32(a, b);  // each half broadcast to all 64 lanes
  x0 = __builtin_bit_cast(float, a);
  x1 = __builtin_bit_cast(float, b);
}

// Transposing LDS read (gfx950 ds_read_b64_tr_b16): the 16 lanes of a group
// pass the addresses of a 4 x 16 block of 16-bit values, lane i the four at
// row i / 4, columns 4 (i % 4) ..; lane i gets column i, rows 0 .. 3.
__device__ __forceinline__ u32x2 lds_read_tr16(const void* p) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p));
}

// Running-max sentinel: a finite stand-in for -inf, so that -max * c stays
// finite and exp2(s * c - max * c) of a masked score (-inf) is exactly 0.
constexpr float M_EMPTY = -1.0e30f;

}  // namespace cab
