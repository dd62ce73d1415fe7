// Common device helpers for the gfx950 (CDNA4, MI355X) kernels.
// Wave64 everywhere: lane = threadIdx.x & 63, reductions span 64 lanes.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define EIA_WAVE 64

typedef __bf16 bf16_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;

#define EIA_DEV __device__ __forceinline__

EIA_DEV float bf2f(bf16_t x) { return (float)x; }
EIA_DEV bf16_t f2bf(float x) { return (bf16_t)x; }   // v_cvt_pk_bf16_f32 (RNE, NaN-safe)

EIA_DEV float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
EIA_DEV float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// Over the sixteen lanes of a row, in all of them (row_ror by 8, 4, 2, 1: no LDS).
#define EIA_ROW_ROR(v, n) \
  __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + (n), 0xf, 0xf, true))
EIA_DEV float row16_sum(float v) {
  v += EIA_ROW_ROR(v, 8);
  v += EIA_ROW_ROR(v, 4);
  v += EIA_ROW_ROR(v, 2);
  return v + EIA_ROW_ROR(v, 1);
}
EIA_DEV float row16_max(float v) {
  v = fmaxf(v, EIA_ROW_ROR(v, 8));
  v = fmaxf(v, EIA_ROW_ROR(v, 4));
  v = fmaxf(v, EIA_ROW_ROR(v, 2));
  return fmaxf(v, EIA_ROW_ROR(v, 1));
}

// Block-wide sum through LDS; `scratch` must hold blockDim.x/64 floats.
EIA_DEV float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  float r = 0.f;
  for (int i = 0; i < nw; ++i) r += scratch[i];
  return r;
}

EIA_DEV float block_max(float v, float* scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  float r = -INFINITY;
  for (int i = 0; i < nw; ++i) r = fmaxf(r, scratch[i]);
  return r;
}

// Error codes returned by the extern "C" launchers (checked by the Python side).
enum EiaStatus : int {
  EIA_OK = 0,
  EIA_BAD_SHAPE = 1001,
  EIA_UNSUPPORTED = 1002,
};

#define EIA_LAUNCH_CHECK() return (int)hipGetLastError()

#define EIA_API extern "C" __attribute__((visibility("default")))

// Element access for kernels templated on the activation type (bf16 or float); math is fp32.
template <typename T> EIA_DEV float ld_f32(const T* p, long i);
template <> EIA_DEV float ld_f32<bf16_t>(const bf16_t* p, long i) { return (float)p[i]; }
template <> EIA_DEV float ld_f32<float>(const float* p, long i) { return p[i]; }
template <typename T> EIA_DEV void st_f32(T* p, long i, float v);
template <> EIA_DEV void st_f32<bf16_t>(bf16_t* p, long i, float v) { p[i] = (bf16_t)v; }
template <> EIA_DEV void st_f32<float>(float* p, long i, float v) { p[i] = v; }

// Four steps of an fp32 matrix-core product (16x16x4): lane l of an A operand holds row l % 16 and
// contraction indices 4 (l / 16) + i, of a B operand column l % 16 and the same indices; the
// accumulator holds rows 4 (l / 16) + i of column l % 16, so that an accumulator is, register by
// register, the B operand of a product over its rows (and the A operand of one over its columns'
// transpose).
EIA_DEV f32x4 mfma_f32_k16(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
  return c;
}

// Stands between matrix products and a branch behind which their results are read by other than a
// matrix product.  Such a read needs up to 12 wait states after the product (32x32x16 bf16; 10 after
// 16x16x4 fp32, 8 after 16x16x32 bf16), which nothing but the instruction stream provides; the compiler
// counts them inside a block but has left out half of them where one way round a branch was short.
// So the wait covers all of it by itself, whatever the code around it becomes.
// All results are operands of the one statement: products of an accumulator that were not could be moved
// behind it.
template <typename V> EIA_DEV void mfma_settle(V& a) { asm volatile("s_nop 11" : "+v"(a)); }
template <typename V> EIA_DEV void mfma_settle(V& a, V& b) { asm volatile("s_nop 11" : "+v"(a), "+v"(b)); }
template <typename V> EIA_DEV void mfma_settle(V (&o)[1]) { mfma_settle(o[0]); }
template <typename V> EIA_DEV void mfma_settle(V (&o)[2]) { mfma_settle(o[0], o[1]); }
template <typename V> EIA_DEV void mfma_settle(V (&o)[4]) {
  asm volatile("s_nop 11" : "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]));
}
template <typename V> EIA_DEV void mfma_settle(V (&o)[8]) {
  asm volatile("s_nop 11" : "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]), "+v"(o[4]), "+v"(o[5]),
               "+v"(o[6]), "+v"(o[7]));
}

// One access from memory straight to LDS: lane i's 16 bytes at gsrc go to byte lds_addr + 16 i.  Not
// counted by the compiler: the caller waits for vmcnt, and for its own reads of the place before.
EIA_DEV void glds16(const void* gsrc, unsigned lds_addr) {
  unsigned keep;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(keep)
      : "v"(gsrc), "s"(__builtin_amdgcn_readfirstlane(lds_addr))
      : "memory");
}
EIA_DEV unsigned lds_offset(const void* p) {
  return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

// Two fp32 numbers as sums of three bf16 ones each, largest part first: 24 bits in three times eight, exact from
// 2^-103 (what is left of smaller numbers for the third part may be flushed) up to bf16's largest, 2^127 (2 - 2^-7).  A
// matrix product of such parts with bf16 operands, or of the six largest pairs of parts, keeps what an fp32
// product keeps at 3/16 or 6/16 of its matrix cycles.  The first part of what rounds past bf16's largest is infinite,
// and parts of what is not finite are no numbers, so callers look for sums that are not finite and form those anew.
EIA_DEV void split3(float a, float b, bf16x2& h, bf16x2& m, bf16x2& l) {
  typedef __attribute__((ext_vector_type(2))) float f32x2_t;
  auto up = [](bf16x2 v, int i) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    return __uint_as_float(i ? u & 0xffff0000u : u << 16);
  };
  h = __builtin_convertvector(f32x2_t{a, b}, bf16x2);
  const float ra = a - up(h, 0), rb = b - up(h, 1);
  m = __builtin_convertvector(f32x2_t{ra, rb}, bf16x2);
  l = __builtin_convertvector(f32x2_t{ra - up(m, 0), rb - up(m, 1)}, bf16x2);
}
EIA_DEV void split3(const float (&v)[8], bf16x8 (&part)[3]) {
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    bf16x2 x[3];
    split3(v[e], v[e + 1], x[0], x[1], x[2]);
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      part[p][e] = x[p][0];
      part[p][e + 1] = x[p][1];
    }
  }
}
EIA_DEV f32x4 mfma_bf16_k32(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// Transposing reads of LDS: lane l of sixteen names row l / 4, entries 4 (l % 4) .. + 3 of a tile of 4 rows
// and 16 columns, and receives its column l.  Two tiles: eight rows of a column, an operand of 16x16x32.
EIA_DEV bf16x8 lds_columns(const bf16_t* p0, const bf16_t* p1) {
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p0);
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p1);
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}
