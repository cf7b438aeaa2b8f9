// Device helpers of the 32x32x16 matrix-core attention kernels (kernels_attn32.hip,
// kernels_attn_nv.hip).
#pragma once

#include "common.hpp"

namespace irodori {

// Max of v over lanes l and l ^ 32 (the two halves of a query column) by v_permlane32_swap,
// a VALU exchange, instead of an LDS-routed shuffle.
__device__ __forceinline__ float max_halves(float v) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__builtin_bit_cast(float, (unsigned)sw[0]), __builtin_bit_cast(float, (unsigned)sw[1]));
}
// Sum of v over lanes l and l ^ 32, the same exchange (the same value in both lanes).
__device__ __forceinline__ float sum_halves(float v) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __builtin_bit_cast(float, (unsigned)sw[0]) + __builtin_bit_cast(float, (unsigned)sw[1]);
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// 8-element operand vector of the 32x32x16 matrix-core step for each element type.
template <typename T>
struct Vec8;
template <>
struct Vec8<bf16> {
    typedef bf16x8 type;
};
template <>
struct Vec8<f16> {
    typedef f16x8 type;
};
__device__ __forceinline__ f32x16 mma32x16(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mma32x16(f16x8 a, f16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ void raw_barrier() { asm volatile("s_barrier" ::: "memory"); }
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, unsigned bytes) {
    // Raw (stride 0) buffer; dword3 0x00020000 is the gfx9-family data format for raw access.
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void buf_load_lds16(__amdgpu_buffer_rsrc_t r, unsigned voff, void* lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, voff, 0, 0, 0);
}
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

}  // namespace irodori
