// Splits of fp32 values into 16-bit planes and the matrix instruction that
// multiplies them, shared by the attention kernels of fp32 accuracy.
//
// Three bf16 planes hold all 24 bits of an fp32 value of at least 2^-110: below,
// the third (then the second) falls under bf16's smallest subnormal, 2^-133
// (the matrix cores keep subnormals), and the value is off by up to 2^-134. The
// kernels see to it that this does not show: probabilities are scaled by 2^16;
// a Q value below 2^-110, or so large that 2^-134 of K would count, and results
// below 2^-100, where 2^-134 of V would, make a query block start over in fp32.
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

// |x| as an integer that orders like it, zero above all others.
__device__ __forceinline__ uint32_t nonzero_magnitude(float x) { return (__builtin_bit_cast(uint32_t, x) << 1) - 1u; }
constexpr uint32_t magnitude_of_exponent(int e) { return ((uint32_t)(e + 127) << 24) - 1u; }

// Whether planes give the scores of queries in full, from the smallest nonzero
// magnitude and the largest absolute value among them: their own planes are
// exact, and an error of 2^-134 in each of 512 values of K moves a score by less
// than 2^-29 log2 units (c: the softmax scale in those units).
__device__ __forceinline__ bool planes_carry_queries(uint32_t smallest, float largest, float c) {
    return smallest >= magnitude_of_exponent(-110) && largest * fmaxf(c, 1.0f) <= 0x1p95f;
}
// Whether results may have lost bits of V.
__device__ __forceinline__ bool results_too_small(uint32_t smallest) { return smallest < magnitude_of_exponent(-100); }

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
