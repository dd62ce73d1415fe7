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
template <typename V> EIA_DEV void mfma_settle(V& a, V& b) { asm volatile("s_nop 11" : "+v"(a), "+v"(b)); }
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
