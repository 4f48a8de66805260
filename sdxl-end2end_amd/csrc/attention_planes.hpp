// Exact splits of fp32 values into 16-bit planes and the matrix instruction
// that multiplies them, shared by the attention kernels of fp32 accuracy.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sdxl_hip {
namespace {

typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <bool kF16>
__device__ __forceinline__ f32x16 mfma32(i16x8 a, i16x8 b, f32x16 c) {
    if constexpr (kF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// A vector conversion: from two scalar ones the compiler converts the low value
// a second time to unpack it (11 instead of 5.5 instructions per split value).
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
}
__device__ __forceinline__ float lo_bf16(uint32_t v) { return __builtin_bit_cast(float, v << 16); }
__device__ __forceinline__ float hi_bf16(uint32_t v) { return __builtin_bit_cast(float, v & 0xFFFF0000u); }

// a less the low (kHi: high) fp16 value of h, in one instruction.
template <bool kHi>
__device__ __forceinline__ float less_f16(float a, uint32_t h) {
    float r;
    if constexpr (kHi) asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(a));
    else asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(a));
    return r;
}

// Two values as kN bf16 or fp16 planes, each holding what the ones before it
// left. fp16 planes before the last are truncated, two values in one
// instruction.
template <int kN, bool kF16>
__device__ __forceinline__ void split2(float a, float b, uint32_t (&out)[kN]) {
#pragma unroll
    for (int i = 0; i < kN; ++i) {
        if constexpr (kF16) {
            if (i + 1 == kN) {
                out[i] = __builtin_bit_cast(uint32_t, f16x2{(_Float16)a, (_Float16)b});
            } else {
                out[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
                a = less_f16<false>(a, out[i]);
                b = less_f16<true>(b, out[i]);
            }
        } else {
            out[i] = pack_bf16(a, b);
            if (i + 1 < kN) {
                a -= lo_bf16(out[i]);
                b -= hi_bf16(out[i]);
            }
        }
    }
}

}  // namespace
}  // namespace sdxl_hip
