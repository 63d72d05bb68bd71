// Shared device helpers for the abridged-KV kernels (gfx950 / CDNA4, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mask_walk.h"

namespace abkv {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Paged cache geometry of the served model (Qwen3-4B attention: 8 KV heads x 128, pages of 16 slots):
// one page of one layer is [2 (K,V)][16 slots][8 heads][128 dims] bf16 = 64 KiB.
constexpr int kPage = 16;
constexpr int kHeadsKV = 8;
constexpr int kHeadDim = 128;
constexpr int kGroup = 4;                                  // query heads per KV head
constexpr int kHeadsQ = kHeadsKV * kGroup;
constexpr int kSlotElems = kHeadsKV * kHeadDim;            // 1024 elements = 2 KiB per slot per K or V
constexpr int kHalfElems = kPage * kSlotElems;             // 16384 elements = 32 KiB (K half of a page)
constexpr int kPageElems = 2 * kHalfElems;                 // 32768 elements = 64 KiB

// Power of two `scale` that brings x (>= 0) into [2^14, 2^15), the top of fp16's range, and its reciprocal: fp16 partials
// keep 11 bits of every value down to 2^-28 of the largest, wherever that lies. (x under 2^-86 keeps the scale of 2^-86.)
struct F16Range {
  float scale, inv;
  __device__ __forceinline__ explicit F16Range(float x) {
    const int e = max((int)(__builtin_bit_cast(uint32_t, x) >> 23) - 14, 27);
    scale = __builtin_bit_cast(float, (uint32_t)e << 23);
    inv = __builtin_bit_cast(float, (uint32_t)(254 - e) << 23);
  }
};

__device__ __forceinline__ floatx4 mfma16x16x32(const bf16x8 a, const bf16x8 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  // v_cvt_pk_bf16_f32: round-to-nearest-even of both halves
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  bf16x2 v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ float xor_shfl(float v, int mask) { return __shfl_xor(v, mask, 64); }

// Reductions over the lane pairs {l, l ^ 16} and {l, l ^ 32} with gfx950's v_permlane16_swap / v_permlane32_swap:
// with both operands = v, the two results hold v[l] and v[l ^ 16] (resp. ^ 32) in some order, so combining them
// reduces the pair in VALU (no LDS round trip).
__device__ __forceinline__ float max_xor16(float v) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float max_xor32(float v) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_xor16(float v) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float sum_xor32(float v) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

}  // namespace abkv
