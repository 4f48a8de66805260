// One query row of online-softmax attention by one wave64, in plain fp32: the
// per-row kernel, and what the tiled kernel falls back to for rows whose
// values it cannot carry.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sdxl_hip {
namespace {

template <typename T>
__device__ __forceinline__ float load_f(const T* p) {
    return (float)(*p);
}

template <typename T>
__device__ __forceinline__ void store_f(T* p, float v) {
    *p = (T)v;
}

__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x = fmaxf(x, __shfl_xor(x, off, 64));
    return x;
}

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    return x;
}

// kChannels: output channels per lane (lane, lane + 64, ...), at least D / 64.
// qs: D floats of LDS of the wave's own. mask: the batch's key mask or null;
// keys from n_keys on are not visible.
template <typename T, int kChannels>
__device__ __forceinline__ void row_attention(const T* qrow, const T* kb, const T* vb, T* orow, int64_t k_stride, int64_t v_stride,
                                              const int32_t* mask, int n_keys, int D, float scale, float* qs) {
    const int lane = threadIdx.x & 63;
    for (int d = lane; d < D; d += 64) qs[d] = load_f(qrow + d);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    const int n_ch = (D + 63) >> 6;
    float acc[kChannels];
#pragma unroll
    for (int t = 0; t < kChannels; ++t) acc[t] = 0.0f;
    float m = -__builtin_inff();
    float l = 0.0f;

    for (int k0 = 0; k0 < n_keys; k0 += 64) {
        const int key = k0 + lane;
        bool visible = key < n_keys;
        if (visible && mask != nullptr) visible = mask[key] != 0;
        float s = -__builtin_inff();
        if (visible) {
            const T* krow = kb + (int64_t)key * k_stride;
            float dot = 0.0f;
            for (int d = 0; d < D; ++d) dot += qs[d] * load_f(krow + d);
            s = dot * scale;
        }
        const float m_new = fmaxf(m, wave_max(s));
        if (m_new == -__builtin_inff()) continue;  // nothing visible yet
        const float alpha = m == -__builtin_inff() ? 0.0f : expf(m - m_new);
        const float pr = visible ? expf(s - m_new) : 0.0f;
        l = l * alpha + wave_sum(pr);
        m = m_new;
        const int chunk = n_keys - k0 < 64 ? n_keys - k0 : 64;
#pragma unroll
        for (int t = 0; t < kChannels; ++t) {
            if (t < n_ch) acc[t] *= alpha;
        }
        for (int j = 0; j < chunk; ++j) {
            const float pj = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, pr), j));
            const T* vrow = vb + (int64_t)(k0 + j) * v_stride;
#pragma unroll
            for (int t = 0; t < kChannels; ++t) {
                const int d = lane + 64 * t;
                if (t < n_ch && d < D) acc[t] += pj * load_f(vrow + d);
            }
        }
    }
    const float inv = 1.0f / fmaxf(l, 1.0e-20f);
#pragma unroll
    for (int t = 0; t < kChannels; ++t) {
        const int d = lane + 64 * t;
        if (t < n_ch && d < D) store_f(orow + d, acc[t] * inv);
    }
}

}  // namespace
}  // namespace sdxl_hip
