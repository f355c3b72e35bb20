// Pieces shared by the MFMA grouped GEMM kernels (gemm.hip, stream.hip).
#pragma once

#include "common.hpp"

namespace uocr {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kXcds = 8;

__device__ __forceinline__ uint16_t bf16_bits(float v) {
  return __builtin_bit_cast(uint16_t, (__bf16)v);
}

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// Eight int8 weights (two words) as bf16: |q| <= 127 is exact in bf16 (the
// f32 of a small integer has zero low half), so the bf16 is its high half.
__device__ __forceinline__ bf16x8 widen_int8x8(uint32_t lo, uint32_t hi) {
  uint32_t p[4];
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    const uint32_t word = j < 4 ? lo : hi;
    const int s0 = 8 * (j & 3), s1 = s0 + 8;
    const float w0 = (float)(int8_t)((word >> s0) & 0xffu);
    const float w1 = (float)(int8_t)((word >> s1) & 0xffu);
    p[j / 2] = __builtin_amdgcn_perm(__float_as_uint(w1), __float_as_uint(w0), 0x07060302u);
  }
  return as_bf16x8(make_uint4(p[0], p[1], p[2], p[3]));
}

constexpr uint32_t kDmaOut = 0x80000000u;  // offset past every resource

// A raw buffer resource over `bytes` bytes from `base` for stores: a store
// whose offset lies past the range is dropped by the hardware range check.
// Row offsets are passed through vgpr_offset, which keeps each whole in the
// VGPR offset (the compiler cannot split a constant part of it into the
// instruction or SGPR offset fields), so the check sees the full row.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t store_rsrc(void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(base, (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ int vgpr_offset(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

}  // namespace uocr
