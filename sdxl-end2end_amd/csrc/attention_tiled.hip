// Tiled attention with 32-bit accuracy for every dtype and head dimension that
// the 16-bit head_dim-64 kernels do not take: FP32 calls, fp16/bf16 at other
// head dimensions, unaligned rows; key masks and causal calls included. Same
// semantics as the per-row kernel (attention_online.hip; reference
// src/cuda/ops_kernels.cu:491-630, :1355-1419).
//
// Arithmetic: the 16-bit matrix cores run 16x the rate of the fp32 ones, so
// fp32 operands are split into three bf16 planes (8 + 8 + 8 significant bits,
// x = h + m + l; attention_planes.hpp) and a product is the six plane products whose weight is
// at least 2^-17 of it (hh, hm, mh, mm, hl, lh); the dropped ones weigh 2^-26,
// below an fp32 rounding. fp16 and bf16 inputs are one plane, exact. The
// probabilities, fp32 in the per-row kernel, keep their bits as planes too:
// three bf16 planes scaled by 2^16 for fp32 and bf16 calls, three fp16 planes by 2^15
// for fp16 calls: all 24 bits of those from 2^-16 of the row's largest on, below
// within 2^-40 of it, which times the largest fp16 value is the smallest one
// ([2, 8, 1000, 80] 30.1 us; two planes, 22 bits, took 27.3). All sums are fp32.
//
// Work split: a workgroup = 4 waves = 4 / kKS blocks of 32 queries x kKS key
// groups. Per stage kKS sub-tiles of 32 keys are loaded (into registers, one
// stage ahead), split once for the whole workgroup and written to LDS as
// planes; a wave then takes one sub-tile for its query block with
// v_mfma_f32_32x32x16: S^T = K Q^T (Q planes in registers), exact running
// maximum, O^T += V^T P^T (V^T by the transposing LDS read, P^T straight from
// the score registers). The key groups of a query block merge through LDS.
//
// Measured (graph replay): FP32 [1, 20, 1024, 64] 1943 us on the per-row kernel,
// 58 us here (92 TFLOP/s; the fp32 matrix cores' peak is 157); FP32
// [2, 8, 1000, 160] 91 us, fp16 [2, 8, 1000, 80] 1676 -> 30.1 us. Against 64 bits
// the FP32 result is closer than the per-row kernel's (4.1e-7 against 6.4e-7 of
// the output's norm at 1024 keys). Per wave and sub-tile 48 MFMAs (1536 cycles)
// meet ~400 other vector instructions (~1600 cycles: the split of the stage's
// share and of the probabilities, the softmax); two waves per SIMD overlap
// them in part. Looking for special values in the results instead of while
// splitting took 4-17 % off every shape (61.3 -> 58.3, 20.8 -> 17.3 us at
// [4, 20, 1024 x 77, 80]).
//
// LDS rows are 64-dim panels of 128 bytes, 16-byte chunks XOR-swizzled by row.
//
// Values that planes cannot carry (infinities, NaN, fp32 above the largest
// bf16; fp32 below 2^-110 where it counts) leave NaN or tiny results; a query block with any starts over in plain
// fp32, its rows dealt to the waves of its key groups (redo_rows).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "attention_kernels.hpp"
#include "attention_planes.hpp"

namespace sdxl_hip {
namespace {

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
typedef __attribute__((address_space(3))) i16x8 lds_i16x8;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;

constexpr int kKeys = 32;                       // keys per sub-tile
constexpr int kPanelBytes = kKeys * 128;        // 32 rows of 64 16-bit values

__device__ __forceinline__ int rev3(int x) { return ((x & 1) << 2) | (x & 2) | ((x >> 2) & 1); }
__device__ __forceinline__ int swz(int row) { return rev3((row >> 1) & 7); }
__device__ __forceinline__ float xhalf_max(float x) { return fmaxf(x, __shfl_xor(x, 32, 64)); }
__device__ __forceinline__ float xhalf_sum(float x) { return x + __shfl_xor(x, 32, 64); }
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

template <typename T> struct Planes;
template <> struct Planes<float> { static constexpr int in = 3, prob = 3; static constexpr bool f16 = false; static constexpr float weight = 65536.0f; };
template <> struct Planes<__bf16> { static constexpr int in = 1, prob = 3; static constexpr bool f16 = false; static constexpr float weight = 65536.0f; };
template <> struct Planes<_Float16> { static constexpr int in = 1, prob = 3; static constexpr bool f16 = true; static constexpr float weight = 32768.0f; };

// Eight values of a row as loaded (fp32: two registers of four; 16-bit: one).
template <typename T> struct Raw { u32x4 v[sizeof(T) == 4 ? 2 : 1]; };

// Values d0 .. d0 + 7 of the row at byte offset off of a uniform base; those
// past the row's n values are others of the row (they meet zero Q values, or
// outputs that are not stored). kVec: n % 8 == 0 and 16-byte aligned.
template <typename T, bool kVec>
__device__ __forceinline__ Raw<T> load8(const char* base, uint32_t off, int d0, int n) {
    Raw<T> r;
    constexpr int kRegs = sizeof(T) == 4 ? 2 : 1;
    if constexpr (kVec) {
        off += (uint32_t)(d0 < n ? d0 : 0) * (uint32_t)sizeof(T);
#pragma unroll
        for (int i = 0; i < kRegs; ++i) r.v[i] = *(const u32x4*)(base + (off + 16u * i));
    } else {
        // an opaque copy keeps the eight offsets from being kept over the stages
        asm volatile("" : "+v"(off));
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int i = 0; i < 8; ++i) r.v[i >> 2][i & 3] = *(const uint32_t*)(base + (off + 4u * (uint32_t)min(d0 + i, n - 1)));
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t lo = *(const uint16_t*)(base + (off + 2u * (uint32_t)min(d0 + 2 * i, n - 1)));
                const uint32_t hi = *(const uint16_t*)(base + (off + 2u * (uint32_t)min(d0 + 2 * i + 1, n - 1)));
                r.v[0][i] = lo | (hi << 16);
            }
        }
    }
    return r;
}

// Planes of eight loaded values (out[plane]).
template <typename T>
__device__ __forceinline__ void planes8(const Raw<T>& r, u32x4 (&out)[Planes<T>::in]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (sizeof(T) == 4) {
            uint32_t w[3];
            split2<3, false>(__builtin_bit_cast(float, (uint32_t)r.v[i >> 1][2 * (i & 1)]),
                             __builtin_bit_cast(float, (uint32_t)r.v[i >> 1][2 * (i & 1) + 1]), w);
#pragma unroll
            for (int pl = 0; pl < 3; ++pl) out[pl][i] = w[pl];
        } else {
            out[0][i] = r.v[0][i];
        }
    }
}

// Zeroes the values from n on of eight.
template <int kN>
__device__ __forceinline__ void zero_past(u32x4 (&pl)[kN], int n) {
    if (n >= 8) return;
#pragma unroll
    for (int i = 0; i < kN; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) pl[i][e] = 2 * e >= n ? 0u : 2 * e + 1 >= n ? pl[i][e] & 0xFFFFu : pl[i][e];
}

// kRedoRows query rows in plain fp32 by one wave, for the blocks whose values
// planes cannot carry: the per-row kernel's steps (attention_online.hip: chunks
// of 64 keys, one key per lane for the scores, one output channel per lane for
// the output), with each K and V value loaded once for all of the rows. In line
// and small, so that it takes no more registers than the kernel around it.
// A NaN in K, so every block here: FP32 [1, 20, 1024, 64] 0.73 ms, fp16 [2, 8, 1000,
// 80] 0.73 (1.94 and 1.67 on the per-row kernel, 8.3 and 11.6 with one row at a
// time by the first wave of a query block alone). q and o point at the first of
// the rows; qs: kRedoRows * dim floats of LDS of the wave's own.
template <typename T, int kRedoRows>
__device__ __forceinline__ void redo_rows(const T* q, const T* k, const T* v, T* o, int64_t q_stride, int64_t k_stride,
                                          int64_t v_stride, int64_t o_stride, const int32_t* mask, int rows, int first_row,
                                          int k_seq, bool causal, int dim, float scale, lds_f32x4* qs) {
    constexpr int kChannels = 3;  // dim <= 160
    const int lane = threadIdx.x & 63;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int d = lane; d < dim; d += 64) {
#pragma unroll
        for (int h = 0; h < kRedoRows / 4; ++h) {
            f32x4 x;
#pragma unroll
            for (int r = 0; r < 4; ++r) x[r] = (float)q[min(4 * h + r, rows - 1) * q_stride + d];
            qs[(kRedoRows / 4) * d + h] = x;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    float acc[kRedoRows][kChannels], m[kRedoRows], l[kRedoRows];
#pragma unroll
    for (int r = 0; r < kRedoRows; ++r) {
        m[r] = -__builtin_inff();
        l[r] = 0.0f;
#pragma unroll
        for (int t = 0; t < kChannels; ++t) acc[r][t] = 0.0f;
    }
    const int n_keys = causal ? min(k_seq, first_row + rows) : k_seq;
#pragma unroll 1
    for (int k0 = 0; k0 < n_keys; k0 += 64) {
        const int key = min(k0 + lane, k_seq - 1);
        const bool shown = k0 + lane < n_keys && (mask == nullptr || mask[key] != 0);
        const T* krow = k + (int64_t)key * k_stride;
        float p[kRedoRows];
#pragma unroll
        for (int r = 0; r < kRedoRows; ++r) p[r] = 0.0f;
#pragma unroll 4
        for (int d = 0; d < dim; ++d) {
            const float x = (float)krow[d];
#pragma unroll
            for (int h = 0; h < kRedoRows / 4; ++h) {
                const f32x4 y = qs[(kRedoRows / 4) * d + h];
#pragma unroll
                for (int r = 0; r < 4; ++r) p[4 * h + r] += y[r] * x;
            }
        }
        int chunk[kRedoRows];  // keys of the chunk that reach the row
#pragma unroll
        for (int r = 0; r < kRedoRows; ++r) {
            const int row_keys = causal ? min(k_seq, first_row + r + 1) : k_seq;
            const bool visible = shown && key < row_keys;
            const float s = visible ? p[r] * scale : -__builtin_inff();
            const float m_new = fmaxf(m[r], wave_max(s));
            const bool none = m_new == -__builtin_inff();  // no finite score yet: the chunk is left out
            const float alpha = m[r] == -__builtin_inff() ? 0.0f : expf(m[r] - m_new);
            p[r] = visible && !none ? expf(s - m_new) : 0.0f;
            l[r] = l[r] * alpha + wave_sum(p[r]);
            m[r] = m_new;
            chunk[r] = none ? 0 : __builtin_amdgcn_readfirstlane(min(64, row_keys - k0));
#pragma unroll
            for (int t = 0; t < kChannels; ++t) acc[r][t] *= alpha;
        }
        const int n = min(64, n_keys - k0);
        for (int j = 0; j < n; ++j) {
            const T* vrow = v + (int64_t)(k0 + j) * v_stride;
            float x[kChannels];
#pragma unroll
            for (int t = 0; t < kChannels; ++t) x[t] = (float)vrow[min(lane + 64 * t, dim - 1)];
#pragma unroll
            for (int r = 0; r < kRedoRows; ++r) {
                const float pj = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p[r]), j));
#pragma unroll
                for (int t = 0; t < kChannels; ++t)
                    if (j < chunk[r]) acc[r][t] += pj * x[t];
            }
        }
    }
#pragma unroll
    for (int r = 0; r < kRedoRows; ++r) {
        const float inv = 1.0f / fmaxf(l[r], 1.0e-20f);
#pragma unroll
        for (int t = 0; t < kChannels; ++t)
            if (r < rows && lane + 64 * t < dim) o[r * o_stride + lane + 64 * t] = (T)(acc[r][t] * inv);
    }
}

constexpr int tiled_panels(int dp) { return (dp + 63) / 64; }
template <typename T>
constexpr int tiled_lds(int dp, int ks) { return 2 * ks * Planes<T>::in * tiled_panels(dp) * kPanelBytes; }

template <typename T>
constexpr int tiled_occupancy(int dp) { return sizeof(T) == 4 ? (dp <= 64 ? 2 : 1) : (dp <= 64 ? 3 : dp <= 128 ? 2 : 1); }

template <typename T, int kDp, int kKS, bool kVec, int kOcc>
__global__ __launch_bounds__(256, kOcc) void tiled_attention_kernel(OnlineAttentionParams p, int q_blocks) {
    constexpr int kIn = Planes<T>::in, kProb = Planes<T>::prob;
    constexpr bool kF16 = Planes<T>::f16;
    constexpr int kPanels = tiled_panels(kDp);
    constexpr int kPlane = kPanels * kPanelBytes;  // one plane of a sub-tile
    constexpr int kSub = kIn * kPlane;             // K or V of a sub-tile
    constexpr int kQB = 4 / kKS;                   // query blocks per workgroup
    constexpr int kSteps = kDp / 16, kTiles = kDp / 32;
    constexpr int kChunks = kDp / 8;               // 8-value chunks per row
    constexpr int kLoads = (kKS * kKeys * kChunks + 255) / 256;
    constexpr int kMergeFloats = kTiles * 16 + 2;
    constexpr int kMergeBytes = (4 - kQB) * kMergeFloats * 64 * 4;
    constexpr int kLdsBytes = 2 * kKS * kSub > kMergeBytes ? 2 * kKS * kSub : kMergeBytes;
    static_assert(kLdsBytes <= 160 * 1024 - 64, "LDS");
    constexpr int kRedoRows = sizeof(T) == 4 || kDp > 64 ? 8 : 4;  // as many as the kernel's registers hold
    static_assert(kRedoRows % 4 == 0 && 4 * kRedoRows * kDp * 4 <= kLdsBytes, "queries of redo_rows");
    __shared__ __attribute__((aligned(16))) char lds[kLdsBytes];
    __shared__ int special[kQB];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int hf = lane >> 5, col = lane & 31;
    const int kg = wave % kKS;

    // each XCD (workgroup ids deal round robin over 8) takes a contiguous range
    const int n_tasks = (int)gridDim.x;
    const int xcd = blockIdx.x & 7, per = n_tasks >> 3, extra = n_tasks & 7;
    const int task = xcd * per + (xcd < extra ? xcd : extra) + (int)(blockIdx.x >> 3);
    const int bh = task / q_blocks;
    // causal calls: the longest query blocks first
    const int qb = p.causal ? q_blocks - 1 - task % q_blocks : task % q_blocks;
    const int h = bh % p.heads, b = bh / p.heads;
    const int D = p.head_dim;
    const int wg_q0 = qb * (32 * kQB);
    const int q0 = wg_q0 + 32 * (wave / kKS);
    const T* qbase = (const T*)p.q + (int64_t)b * p.q_seq * p.q_row_stride + (int64_t)h * D;
    const T* kbase = (const T*)p.k + (int64_t)b * p.k_seq * p.k_row_stride + (int64_t)h * D;
    const T* vbase = (const T*)p.v + (int64_t)b * p.k_seq * p.v_row_stride + (int64_t)h * D;
    T* obase = (T*)p.o + (int64_t)b * p.q_seq * p.o_row_stride + (int64_t)h * D;

    int n_keys = p.k_seq;
    if (p.causal) n_keys = min(n_keys, wg_q0 + 32 * kQB);
    const int n_stages = (n_keys + kKS * kKeys - 1) / (kKS * kKeys);

    // Q planes: lane holds query q0 + col, dims 16 ks + 8 hf .. +7.
    const int my_query = q0 + col;
    i16x8 qop[kIn][kSteps];
    const float c = p.scale * 1.4426950408889634f;
    uint32_t q_smallest = ~0u;
    float q_largest = 0.0f;
    {
        const uint32_t off = (uint32_t)min(my_query - wg_q0, p.q_seq - 1 - wg_q0) * (uint32_t)(p.q_row_stride * (int64_t)sizeof(T));
        const char* src = (const char*)(qbase + (int64_t)wg_q0 * p.q_row_stride);
#pragma unroll
        for (int ks = 0; ks < kSteps; ++ks) {
            const int d0 = 16 * ks + 8 * hf;
            const Raw<T> r = load8<T, kVec>(src, off, d0, D);
            if constexpr (sizeof(T) == 4)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float x = __builtin_bit_cast(float, (uint32_t)r.v[i >> 2][i & 3]);
                    q_smallest = min(q_smallest, nonzero_magnitude(x));
                    q_largest = fmaxf(q_largest, fabsf(x));
                }
            u32x4 pl[kIn];
            planes8<T>(r, pl);
            zero_past<kIn>(pl, D - d0);
#pragma unroll
            for (int i = 0; i < kIn; ++i) qop[i][ks] = __builtin_bit_cast(i16x8, pl[i]);
        }
    }
    const bool q_carried = __builtin_amdgcn_ballot_w64(!planes_carry_queries(q_smallest, q_largest, c)) == 0;

    // Stage loads: chunk n of the stage is row n / kChunks (sub-tile row / 32),
    // dims 8 (n % kChunks) .. +7.
    Raw<T> kraw[kLoads], vraw[kLoads];
    int mask_word = 1;
    const uint32_t k_stride_b = (uint32_t)(p.k_row_stride * (int64_t)sizeof(T));
    const uint32_t v_stride_b = (uint32_t)(p.v_row_stride * (int64_t)sizeof(T));
    auto load_stage = [&](int s) __attribute__((always_inline)) {
        const int key0 = s * kKS * kKeys;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int n = threadIdx.x + 256 * i;
            const int row = min(n / kChunks, p.k_seq - 1 - key0), d0 = 8 * (n % kChunks);
            kraw[i] = load8<T, kVec>((const char*)(kbase + (int64_t)key0 * p.k_row_stride), (uint32_t)row * k_stride_b, d0, D);
            vraw[i] = load8<T, kVec>((const char*)(vbase + (int64_t)key0 * p.v_row_stride), (uint32_t)row * v_stride_b, d0, D);
        }
        if (p.key_mask != nullptr)
            mask_word = p.key_mask[(int64_t)b * p.k_seq + min(key0 + kKeys * kg + col, p.k_seq - 1)];
    };
    auto write_stage = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int n = threadIdx.x + 256 * i;
            const int srow = n / kChunks, chunk = n % kChunks;
            if (kKS * kKeys * kChunks % 256 == 0 || srow < kKS * kKeys) {
                const int row = srow % kKeys;
                char* dst = lds + (srow / kKeys) * (2 * kSub) + (chunk >> 3) * kPanelBytes + row * 128 + (((chunk & 7) ^ swz(row)) << 4);
                u32x4 pl[kIn];
                planes8<T>(kraw[i], pl);
                // K past D: what load8 put there is the row's own, but an
                // infinity among it would meet Q's zeros (FP32: planes make it NaN)
                if (kIn == 1 && D != kDp) zero_past<kIn>(pl, D - 8 * chunk);
#pragma unroll
                for (int j = 0; j < kIn; ++j) *(lds_u32x4*)(dst + j * kPlane) = pl[j];
                planes8<T>(vraw[i], pl);
#pragma unroll
                for (int j = 0; j < kIn; ++j) *(lds_u32x4*)(dst + kSub + j * kPlane) = pl[j];
            }
        }
    };

    // Operand offsets in a panel: K row col, chunk (2 (ks & 3) + hf) ^ swz(col);
    // V^T by transposing reads (lane r = 4j + qd of each 16 gives key row
    // 4 hf + j, + 8 for the second read, dims 32 dt + 16 ((lane >> 4) & 1) + 4 qd).
    const int k_swz = swz(col);
    int v_off[2][2];
    {
        const int g16 = lane & 15;
        const int key = 4 * hf + (g16 >> 2), qd = g16 & 3;
#pragma unroll
        for (int dt = 0; dt < 2; ++dt) {
            const int chunk = 4 * dt + 2 * ((lane >> 4) & 1) + (qd >> 1);
#pragma unroll
            for (int hi = 0; hi < 2; ++hi)
                v_off[dt][hi] = (key + 8 * hi) * 128 + ((chunk ^ swz(key + 8 * hi)) << 4) + ((qd & 1) << 3);
        }
    }

    f32x16 acc[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.0f;
    float m_run = -__builtin_inff(), l_run = 0.0f;  // log2 units; this lane's half of the sum
    const char* const ksub = lds + kg * (2 * kSub);
    const char* const vsub = ksub + kSub;

    if (n_stages > 0) load_stage(0);
    for (int s = 0; s < n_stages; ++s) {
        __syncthreads();  // stage s - 1 consumed
        const int key0 = s * kKS * kKeys + kKeys * kg;  // this wave's keys
        uint32_t vis = ~0u;
        if (p.key_mask != nullptr) vis = (uint32_t)__builtin_amdgcn_ballot_w64(mask_word != 0);
        if (key0 + kKeys > p.k_seq) vis = key0 < p.k_seq ? vis & ((1u << (p.k_seq - key0)) - 1u) : 0u;
        write_stage();
        __syncthreads();
        if (s + 1 < n_stages) load_stage(s + 1);
        // nothing visible to any of the wave's queries
        if (vis == 0u || (p.causal && key0 > q0 + 31)) continue;

        f32x16 sc;
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[i] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < kSteps; ++ks) {
            const char* src = ksub + (ks >> 2) * kPanelBytes + col * 128 + (((2 * (ks & 3) + hf) ^ k_swz) << 4);
            i16x8 kop[kIn];
#pragma unroll
            for (int i = 0; i < kIn; ++i) kop[i] = *(const lds_i16x8*)(src + i * kPlane);
#pragma unroll
            for (int i = kIn - 1; i >= 0; --i)
#pragma unroll
                for (int j = kIn - 1 - i; j >= 0; --j) sc = mfma32<kF16>(kop[i], qop[j][ks], sc);
        }

        if (vis != ~0u || (p.causal && key0 + 31 > q0)) {
            const uint32_t lane_vis = vis >> (4 * hf);
            const int lim = p.causal ? my_query - key0 - 4 * hf : 0x7FFFFFFF;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int kk = 8 * (i >> 2) + (i & 3);
                sc[i] = ((lane_vis >> kk) & 1u) && kk <= lim ? sc[i] : -__builtin_inff();
            }
        }
        float mx = -__builtin_inff();
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sc[i]);
        mx = xhalf_max(mx) * c;
        if (__builtin_amdgcn_ballot_w64(mx > m_run) != 0) {
            const float m_new = fmaxf(m_run, mx);
            const float alpha = m_run == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            l_run *= alpha;
#pragma unroll
            for (int t = 0; t < kTiles; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[t][i] *= alpha;
        }
        const float shift = m_run == -__builtin_inff() ? 0.0f : -m_run;
        f32x16 pr;
#pragma unroll
        for (int i = 0; i < 16; ++i) pr[i] = Planes<T>::weight * __builtin_amdgcn_exp2f(__builtin_fmaf(sc[i], c, shift));
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(fabsf(m_run) <= 1.0e6f)) != 0, 0)) {
            // no finite score yet (zero weights, as if not visible), or a
            // maximum so large that its own product with c rounds by more than
            // a few units: subtract the rounded products instead
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                float x = sc[i] * c;
                asm("" : "+v"(x));  // rounded: no fused multiply-add
                x -= m_run;
                // a NaN that came with no finite score must still reach the check below
                if (m_run == -__builtin_inff() && sc[i] != sc[i]) l_run = sc[i];
                pr[i] = m_run == -__builtin_inff() ? 0.0f : fabsf(m_run) <= 1.0e6f ? pr[i] : Planes<T>::weight * __builtin_amdgcn_exp2f(x);
            }
        }
#pragma unroll
        for (int i = 0; i < 16; i += 4) l_run += (pr[i] + pr[i + 1]) + (pr[i + 2] + pr[i + 3]);

#pragma unroll
        for (int ss = 0; ss < 2; ++ss) {
            i16x8 pop[kProb];
            {
                uint32_t w[4][kProb];
#pragma unroll
                for (int i = 0; i < 4; ++i) split2<kProb, kF16>(pr[8 * ss + 2 * i], pr[8 * ss + 2 * i + 1], w[i]);
#pragma unroll
                for (int pl = 0; pl < kProb; ++pl) pop[pl] = __builtin_bit_cast(i16x8, u32x4{w[0][pl], w[1][pl], w[2][pl], w[3][pl]});
            }
#pragma unroll
            for (int t = 0; t < kTiles; ++t) {
                i16x8 vop[kIn];
#pragma unroll
                for (int i = 0; i < kIn; ++i) {
                    const char* src = vsub + i * kPlane + (t >> 1) * kPanelBytes + 16 * ss * 128;
                    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(src + v_off[t & 1][0]));
                    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(src + v_off[t & 1][1]));
                    vop[i] = i16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                }
#pragma unroll
                for (int i = kIn - 1; i >= 0; --i)
#pragma unroll
                    for (int j = (kIn == 3 ? 2 - i : kProb - 1); j >= 0; --j) acc[t] = mfma32<kF16>(vop[i], pop[j], acc[t]);
            }
        }
    }

    // merge the key groups of a query block (fixed order) in its first wave
    float l_tot = xhalf_sum(l_run);
    if constexpr (kKS > 1) {
        __syncthreads();
        float* park = (float*)lds + ((wave / kKS) * (kKS - 1) - 1) * (kMergeFloats * 64) + lane;
        if (kg > 0) {
            float* mine = park + kg * (kMergeFloats * 64);
#pragma unroll
            for (int t = 0; t < kTiles; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) mine[(16 * t + i) * 64] = acc[t][i];
            mine[16 * kTiles * 64] = m_run;
            mine[(16 * kTiles + 1) * 64] = l_tot;
        }
        __syncthreads();
#pragma unroll 1
        for (int g = 1; g < (kg == 0 ? kKS : 0); ++g) {
            const float* part = park + g * (kMergeFloats * 64);
            const float m1 = part[16 * kTiles * 64];
            const float mx = fmaxf(m_run, m1);
            const float a0 = m_run == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(m_run - mx);
            const float a1 = m1 == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(m1 - mx);
            m_run = mx;
            l_tot = l_tot * a0 + part[(16 * kTiles + 1) * 64] * a1;
#pragma unroll
            for (int t = 0; t < kTiles; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[t][i] = acc[t][i] * a0 + part[(16 * t + i) * 64] * a1;
        }
    }

    const float inv = 1.0f / fmaxf(l_tot, 1.0e-20f);
    // Planes turn an infinity, a NaN or an FP32 value above the largest bf16
    // into a NaN, which reaches every score or output that it meets: a query
    // block with one (or whose results overflow, or are so small that planes
    // may have lost bits of them) starts over in fp32.
    float bad = l_tot;
    uint32_t smallest = ~0u;
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            acc[t][i] *= inv;
            bad = __builtin_fmaf(acc[t][i], 0.0f, bad);
            if constexpr (sizeof(T) == 4) smallest = min(smallest, nonzero_magnitude(acc[t][i]));
        }
    if (kg == 0) special[wave / kKS] = !q_carried || __builtin_amdgcn_ballot_w64(results_too_small(smallest) || bad != bad) != 0;
    __syncthreads();  // also: nobody reads the tiles or the parked sums any more
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(special[wave / kKS]) != 0, 0)) {
#pragma unroll 1
        for (int r = q0 + kRedoRows * kg; r < min(q0 + 32, p.q_seq); r += kRedoRows * kKS)
            redo_rows<T, kRedoRows>(qbase + (int64_t)r * p.q_row_stride, kbase, vbase, obase + (int64_t)r * p.o_row_stride, p.q_row_stride,
                         p.k_row_stride, p.v_row_stride, p.o_row_stride, p.key_mask != nullptr ? p.key_mask + (int64_t)b * p.k_seq : nullptr,
                         min(kRedoRows, p.q_seq - r), r, p.k_seq, p.causal != 0, D, p.scale, (lds_f32x4*)lds + wave * (kRedoRows / 4 * kDp));
        return;
    }
    if (kg > 0) return;
    if (my_query >= p.q_seq) return;
    T* orow = obase + (int64_t)my_query * p.o_row_stride;
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int d0 = 32 * t + 8 * u + 4 * hf;
            T w[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = (T)acc[t][4 * u + e];
            if constexpr (kVec) {
                if (d0 < D) {
                    if constexpr (sizeof(T) == 4) *(f32x4*)(orow + d0) = f32x4{(float)w[0], (float)w[1], (float)w[2], (float)w[3]};
                    else *(u32x2*)(orow + d0) = __builtin_bit_cast(u32x2, w);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (d0 + e < D) orow[d0 + e] = w[e];
            }
        }
}

template <typename T, int kDp, int kKS, bool kVec, int kOcc = tiled_occupancy<T>(kDp)>
hipError_t launch_one(const OnlineAttentionParams& p, hipStream_t stream) {
    constexpr int kRows = 128 / kKS;
    const int64_t q_blocks = ((int64_t)p.q_seq + kRows - 1) / kRows;
    const int64_t grid = q_blocks * p.heads * p.batch;
    if (grid > 0xFFFFFFFFll / 256) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL((tiled_attention_kernel<T, kDp, kKS, kVec, kOcc>), dim3((unsigned)grid), dim3(256), 0, stream, p, (int)q_blocks);
    return hipGetLastError();
}

// Key groups per workgroup. Two (64 queries share a stage's split) is the
// general choice: the FP32 [1, 20, 1024, 64] call took 64 us with two, 73 with
// one; fp16 [2, 8, 1000, 80] 29.5 with two, 47 with one. One (128 queries) for
// short key sequences on full grids, where a wave has few sub-tiles to merge
// (fp16 [4, 20, 1024 x 77, 80] 19.5 against 21.9 us). Four (32 queries) for
// 16-bit calls of at most two 32-query blocks per CU, whose stages still fit
// (fp16 [1, 4, 100 x 400, 80] 12.1 against 14.0 us, [2, 8, 600, 40] 15.9 against
// 17.1; at 512 blocks, [2, 8, 1000, 128], 50 against 36). Rows that are not
// 16-byte aligned use two.
template <typename T, int kDp>
hipError_t launch_dp(const OnlineAttentionParams& p, int compute_units, bool vec, hipStream_t stream) {
    if (!vec) return launch_one<T, kDp, 2, false>(p, stream);
    const int64_t cus = compute_units > 0 ? compute_units : 256;
    const int64_t blocks = ((int64_t)p.q_seq + 31) / 32 * p.heads * p.batch;
    if constexpr (sizeof(T) == 2) {
        if (p.k_seq > 2 * kKeys && blocks < 2 * cus) return launch_one<T, kDp, 4, true>(p, stream);
    }
    if (p.k_seq <= kKeys || (p.k_seq <= 4 * kKeys && blocks >= 8 * cus)) return launch_one<T, kDp, 1, true>(p, stream);
    // FP32 with more than two workgroups per CU: three waves per SIMD in place
    // of two, although their registers spill ([1, 10, 4096, 64] 330 -> 294 us,
    // [2, 20, 1024, 64] 89.7 -> 81.8, [2, 20, 900, 48] 83 -> 74); with two at
    // most it loses ([2, 16, 1000, 64], exactly two, 58.6 -> 63.1).
    if constexpr (sizeof(T) == 4 && kDp == 64) {
        const int64_t workgroups = ((int64_t)p.q_seq + 63) / 64 * p.heads * p.batch;
        if (workgroups > 2 * cus) return launch_one<T, kDp, 2, true, 3>(p, stream);
    }
    return launch_one<T, kDp, 2, true>(p, stream);
}

template <typename T>
hipError_t launch_type(const OnlineAttentionParams& p, int compute_units, hipStream_t stream) {
    const int64_t e = sizeof(T);
    auto a16 = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
    const bool vec = p.head_dim % 8 == 0 && p.q_row_stride * e % 16 == 0 && p.k_row_stride * e % 16 == 0 &&
                     p.v_row_stride * e % 16 == 0 && p.o_row_stride * e % 16 == 0 && a16(p.q) && a16(p.k) && a16(p.v) && a16(p.o);
    if (p.head_dim <= 32) return launch_dp<T, 32>(p, compute_units, vec, stream);
    if (p.head_dim <= 64) return launch_dp<T, 64>(p, compute_units, vec, stream);
    if (p.head_dim <= 96) return launch_dp<T, 96>(p, compute_units, vec, stream);
    if (p.head_dim <= 128) return launch_dp<T, 128>(p, compute_units, vec, stream);
    return launch_dp<T, 160>(p, compute_units, vec, stream);
}

}  // namespace

// Few queries against few keys leave most of a 64-query tile empty: with at
// least eight (batch, head) pairs per CU the per-row kernel is the faster one as
// long as it has few keys in all to walk per pair, a row counting as six more.
// Measured, tiled against per-row kernel, 2048 pairs, FP32 (line at 90): 1 x 40
// head_dim 40 28.7 / 21.6 us, 160 115 / 52; 4 x 16 20.6 / 19.1, 82 / 55; 1 x 77 41
// / 44, 149 / 99; 4 x 40 29.5 / 47.5, 117 / 108; 16 x 4 21 / 36, 84 / 86; fp16 (line at 40): 1 x 16
// 11.7 / 9.0, 23.9 / 15.6; 4 x 4 11.6 / 10.6, 24.0 / 16.4; 1 x 40 16.2 / 15.9, 33 /
// 43. FP32 calls of at most four keys also on grids that the per-row kernel
// fills only once (4 x 4, 512 pairs 8.1 / 5.8 and 20.6 / 8.8; 16 pairs 6.2 / 5.5 and
// 10.6 / 7.8).
static bool few_enough_for_rows(const OnlineAttentionParams& p, bool fp32, int compute_units) {
    const int64_t cus = compute_units > 0 ? compute_units : 256;
    const int64_t pairs = (int64_t)p.heads * p.batch, rows = pairs * p.q_seq;
    if (rows >= int64_t{1} << 26) return false;  // more workgroups of four rows than a grid holds
    if (pairs >= 8 * cus && (int64_t)p.q_seq * ((int64_t)p.k_seq + 6) <= (fp32 ? 90 : 40)) return true;
    return fp32 && p.k_seq <= 4 && rows <= 8 * cus;
}

bool tiled_attention_eligible(const OnlineAttentionParams& p, int dtype, int compute_units) {
    if (few_enough_for_rows(p, dtype == 2, compute_units)) return false;
    // 32-bit row offsets within a stage of at most 128 rows
    const int64_t limit = int64_t{1} << 23;
    // a grid dimension holds fewer than 2^32 threads (the caller splits batches;
    // large grids take 64 queries per workgroup or more)
    const int64_t workgroups = ((int64_t)p.q_seq + 63) / 64 * p.heads * p.batch;
    return workgroups <= 0xFFFFFFFFll / 256 && dtype >= 0 && dtype <= 2 && p.head_dim <= 160 && p.k_seq > 0 &&
           p.q_row_stride < limit && p.k_row_stride < limit && p.v_row_stride < limit;
}

hipError_t launch_tiled_attention(const OnlineAttentionParams& p, int dtype, int compute_units, hipStream_t stream) {
    if (p.batch == 0 || p.q_seq == 0) return hipSuccess;
    switch (dtype) {
    case 0: return launch_type<_Float16>(p, compute_units, stream);
    case 1: return launch_type<__bf16>(p, compute_units, stream);
    default: return launch_type<float>(p, compute_units, stream);
    }
}

}  // namespace sdxl_hip
