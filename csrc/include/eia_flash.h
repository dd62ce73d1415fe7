// Shared by the 32x32x16 prefill attention kernels (window_flash.hip, latent_flash.hip): a lane owns
// one query row as a column of S^T and O^T, together with lane ^ 32.
#pragma once
#include "eia_common.h"

typedef __attribute__((ext_vector_type(16))) float f32x16_t;

constexpr float FLASH_LOG2E = 1.4426950408889634f;
constexpr float FLASH_DEFER = 8.f;          // log2 by which a tile may exceed the running maximum

EIA_DEV float flash_pair_max(float v) {     // with lane ^ 32
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
EIA_DEV float flash_pair_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// Over the four lanes of a column of a 16 x 16 tile (those with the same lane % 16), in all of them: quarters and
// halves of the wave change places in registers, where shuffles over 16 and 32 lanes wait for LDS.
EIA_DEV float column_max(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return flash_pair_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}
EIA_DEV float column_sum(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return flash_pair_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}
EIA_DEV bf16x2 flash_pack(float a, float b) {          // one v_cvt_pk_bf16_f32
  typedef __attribute__((ext_vector_type(2))) float f32x2_t;
  return __builtin_convertvector(f32x2_t{a, b}, bf16x2);
}

// fp32 weights as bf16 operands: a high part and the remainder.
EIA_DEV void flash_split(float p0, float p1, int j, bf16x8& hi, bf16x8& lo) {
  const bf16x2 h = flash_pack(p0, p1);
  const unsigned hb = __builtin_bit_cast(unsigned, h);
  const bf16x2 l = flash_pack(p0 - __uint_as_float(hb << 16), p1 - __uint_as_float(hb & 0xffff0000u));
  hi[j] = h[0];
  hi[j + 1] = h[1];
  lo[j] = l[0];
  lo[j + 1] = l[1];
}
