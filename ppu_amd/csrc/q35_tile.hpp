// Helpers of the tiled matrix-core kernels: copies from memory straight into
// LDS, explicit waits, the 32 x 32 MFMAs.
#pragma once
#include "q35_common.hpp"

namespace {

typedef __attribute__((address_space(3))) uint8_t lds_u8;
Q35_DEV uint32_t lds_offset(const void* p) { return (uint32_t)(uintptr_t)(const lds_u8*)p; }

// One wave instruction of a stage copy: lane i copies the 16 bytes at
// sbase + voff to LDS bytes [lds + 16 i, +16) (the LDS base goes in m0).
Q35_DEV void dma16(uint32_t lds, const uint8_t* sbase, uint32_t voff) {
  asm volatile("global_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(sbase), "{m0}"(lds) : "memory");
}
// s_waitcnt vmcnt(N) (gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt
// and lgkmcnt at their "no wait" maxima). As a builtin the compiler's wait
// pass sees it and keeps it; it does not know of the asm loads it waits for.
template <int N>
Q35_DEV void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
// This wave's LDS reads complete (s_waitcnt lgkmcnt(0)).
Q35_DEV void wait_lds() { __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (3 << 14)); }
// Keeps the compiler's scheduler from moving any instruction across it.
#define Q35_PIN() __builtin_amdgcn_sched_barrier(0)

typedef float q35_f32x16 __attribute__((ext_vector_type(16)));
typedef int q35_i32x16 __attribute__((ext_vector_type(16)));
typedef int q35_i32x4 __attribute__((ext_vector_type(4)));
Q35_DEV q35_f32x16 mfma32(const q35_u32x4 a, const q35_u32x4 b, q35_f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(q35_bf16x8, a),
                                                 __builtin_bit_cast(q35_bf16x8, b), c, 0, 0, 0);
}
Q35_DEV q35_i32x16 mfma32(const q35_u32x4 a, const q35_u32x4 b, q35_i32x16 c) {
  return __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(q35_i32x4, a),
                                               __builtin_bit_cast(q35_i32x4, b), c, 0, 0, 0);
}

// Lane l and lane l ^ 32: the larger of the two, their sum.
Q35_DEV float half_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
Q35_DEV float half_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

}  // namespace
