// A 16-token tile of decode attention on the matrix cores: the two products, the lane groups' reductions and the V image in LDS
// (shared by attn_decode.hip and attn_decode_small.hip).
#pragma once
#include <type_traits>

#include "common.h"

namespace msgl {

typedef uint32_t V4 __attribute__((ext_vector_type(4)));
constexpr float kNegBig = -3.0e38f;

typedef __attribute__((ext_vector_type(8))) __bf16 dbf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 df16x8;
typedef __attribute__((ext_vector_type(4))) _Float16 df16x4;
typedef __attribute__((ext_vector_type(4))) short ds16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) ds16x4 lds_ds16x4;
typedef __attribute__((address_space(3))) char dlds_char;

template <typename T>
__device__ __forceinline__ f32x4 mfma_k32(const V4& a, const V4& b, f32x4 c) {
  if constexpr (std::is_same_v<T, BF16>)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dbf16x8, a), __builtin_bit_cast(dbf16x8, b), c, 0,
                                                   0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(df16x8, a), __builtin_bit_cast(df16x8, b), c, 0, 0,
                                                  0);
}
template <typename T>
__device__ __forceinline__ f32x4 mfma_k16(const uint2& a, const uint2& b, f32x4 c) {
  if constexpr (std::is_same_v<T, BF16>)
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(ds16x4, a), __builtin_bit_cast(ds16x4, b), c, 0, 0,
                                                     0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(df16x4, a), __builtin_bit_cast(df16x4, b), c, 0, 0, 0);
}

// max over the four 16-lane groups (every lane ends with it)
__device__ __forceinline__ float max_over_rows(float x) {
  const uint32_t u = __float_as_uint(x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const uint32_t w = __float_as_uint(x);
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float sum_over_rows(float x) {
  const uint32_t u = __float_as_uint(x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const uint32_t w = __float_as_uint(x);
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// V image: [16 tokens][256 B]; 64-B blocks XORed by the token's low two bits, the 32-B half by bit 2: the 32 lanes
// of one ds_read_b64_tr_b16 pass (16 lanes x 2 groups) then cover 32 distinct 8-B bank pairs
__device__ __forceinline__ int vimg_off(int tok, int byte_in_row) {
  return tok * 256 + (byte_in_row ^ ((tok & 3) << 6) ^ (((tok >> 2) & 1) << 5));
}

}  // namespace msgl
