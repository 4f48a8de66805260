// FP32 attention at head dimension 512.
//
// The SDXL VAE decoder's mid-block attention is single-head with the head
// width equal to the 512 channels, in FP32 (reference src/cuda/vae.cpp:65-99,
// dispatched to generic_online_attention_f32_kernel,
// src/cuda/ops_kernels.cu:1355-1419: one block per query, keys one by one).
// At a 128x128 latent that is 16384 tokens: 550 GFLOP per call. Same semantics
// (softmax with a running maximum, output divided by max(sum, 1e-20));
// non-causal, unmasked calls with 16-byte aligned rows.
//
// Arithmetic: operands are split into three bf16 planes and a product is six
// plane products on the bf16 matrix cores (attention_planes.hpp), 2.7x
// the fp32 matrix cores' rate; all sums are fp32.
//
// Work split: a workgroup = 8 waves = 32 kQT queries of one (batch, head);
// wave w owns dims 64 w .. +63 of the scores for all of the queries: its slice
// of Q as planes in registers (kQT = 2: the third plane in LDS) and of K,
// which, like its 32 kDT dims of V, comes straight from global memory in the
// matrix operands' layout, so that each element is split by one wave only.
// With kDT = 1 two workgroups share a query block, each with half of the
// output's dims. Per block of 32 keys t:
//   * the partial scores S^T over the wave's 64 dims, formed one block ahead,
//     meet in LDS; each wave sums the eight partials of 4 kQT queries (lane
//     groups of 16 / kQT lanes share a query, its maximum and sum are DPP
//     reductions), forms their probabilities once, and leaves them in LDS as
//     planes, with the factor by which the maximum's move scales O;
//   * meanwhile the waves form the partial scores of block t + 1;
//   * O^T[d][q] += V^T P^T for the wave's output dims.
// Two barriers per block. Each stage of a block is the matrix instructions of
// one operand (12 or 6) with the split of the next operand and the stage's
// share of the other work issued between them: the waves of a SIMD run in
// step, and with the splits in front of the matrix instructions neither unit
// worked while the other did (3.33 against 2.73 ms at 16384 tokens).
//
// Bound: at 64 queries the bf16 matrix cores, busy 72 % of a block's ~8500
// cycles at a power-limited ~1.7 GHz (1.25 PFLOP/s of plane products; the
// vendor's bf16 GEMM reaches 1.16 on the same card); at 32 the split's vector
// instructions and the exchange of the partials (MFMA 3072 of ~6800 cycles).
// Measured against fp32 matrix instructions (v_mfma_f32_32x32x2, the same
// outputs within 64-bit error 2.0e-6 here, 2.3e-6 there): 16384 tokens 5.02 ->
// 2.65 ms (208 TFLOP/s), 8192 1.43 -> 0.86, 4096 0.403 -> 0.342 (two
// workgroups per block; one: 0.400), 1024 105 -> 83 us. Tried and not kept:
// the residuals x - h by v_dot2 (fewer instructions, but wait states: 2.92
// ms), K loads of 64-byte row segments exchanged by v_permlane16_swap (4096
// tokens 421 -> 435 us).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "attention_kernels.hpp"
#include "attention_planes.hpp"

namespace sdxl_hip {
namespace {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
typedef __attribute__((address_space(3))) f32x2 lds_f32x2;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) float lds_float;

constexpr int kDim = 512;
constexpr int kKeys = 32;   // keys per block
constexpr int kWaves = 8;
constexpr int kSlice = 64;  // dims per wave

template <int kCtrl>
__device__ __forceinline__ float dpp(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), kCtrl, 0xF, 0xF, true));
}
// Maximum and sum over groups of 8 (kN = 8) or 16 consecutive lanes, in all of them.
template <int kN>
__device__ __forceinline__ float group_max(float x) {
    x = fmaxf(x, dpp<0xB1>(x));   // quad_perm 1,0,3,2
    x = fmaxf(x, dpp<0x4E>(x));   // quad_perm 2,3,0,1
    x = fmaxf(x, dpp<0x141>(x));  // row_half_mirror
    if constexpr (kN == 16) x = fmaxf(x, dpp<0x140>(x));  // row_mirror
    return x;
}
template <int kN>
__device__ __forceinline__ float group_sum(float x) {
    x += dpp<0xB1>(x);
    x += dpp<0x4E>(x);
    x += dpp<0x141>(x);
    if constexpr (kN == 16) x += dpp<0x140>(x);
    return x;
}

// Whether every one of the workgroup's queries, or any key, holds a NaN: all of
// the workgroup's results are NaN then, as they stand. flags: two zeros in LDS.
__device__ __forceinline__ bool all_rows_nan(const float* q, const float* k, int64_t q_stride, int64_t k_stride, int rows, int k_seq,
                                             volatile __attribute__((address_space(3))) int* flags) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    auto row_nan = [&](const float* row) __attribute__((always_inline)) {
        const f32x4 x = *(const f32x4*)(row + 4 * lane), y = *(const f32x4*)(row + 256 + 4 * lane);
        return __builtin_isunordered(x[0], x[1]) || __builtin_isunordered(x[2], x[3]) || __builtin_isunordered(y[0], y[1]) ||
               __builtin_isunordered(y[2], y[3]);
    };
#pragma unroll 1
    for (int r = wave; r < rows; r += kWaves)
        if (__builtin_amdgcn_ballot_w64(row_nan(q + (int64_t)r * q_stride)) == 0) flags[0] = 1;
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(flags[0]) == 0) return true;
#pragma unroll 1
    for (int key0 = 8 * wave; key0 < k_seq && flags[1] == 0; key0 += 8 * kWaves) {
        bool nan = false;
#pragma unroll
        for (int r = 0; r < 8; ++r) nan = row_nan(k + (int64_t)min(key0 + r, k_seq - 1) * k_stride) || nan;
        if (__builtin_amdgcn_ballot_w64(nan) != 0) flags[1] = 1;
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(flags[1]) != 0;
}

// The output of 32 queries from the start on v_mfma_f32_32x32x2, for calls whose
// values planes cannot carry: the same split over waves and exchange of
// partials, without the pipeline. A NaN score makes its row NaN. q and o point
// at the first query of the rows left, v and o at the wave's first output dim.
// An infinity in K: 16384 tokens 10.7 ms in all (fp32 matrix instructions
// throughout took 5.0, plain rows by a wave each 282), 4096 tokens 1.16 (0.40,
// 35); a NaN in K, by all_rows_nan, 2.7 and 0.37.
template <int kDT>
__device__ __forceinline__ void redo_block(const float* q, const float* k, const float* v, float* o, int64_t q_stride, int64_t k_stride,
                                           int64_t v_stride, int64_t o_stride, int rows, int k_seq, float scale, lds_f32x4* part) {
    const int lane = threadIdx.x & 63, hf = lane >> 5, col = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    f32x4 qx[kSlice / 8], kx[kSlice / 8];  // lane holds query or key col, dims 8 n + 4 hf .. +3 of the slice
    const float* qrow = q + (int64_t)min(col, rows - 1) * q_stride + kSlice * wave + 4 * hf;
    auto load_k = [&](int key0) __attribute__((always_inline)) {
        const float* krow = k + (int64_t)min(key0 + col, k_seq - 1) * k_stride + kSlice * wave + 4 * hf;
#pragma unroll
        for (int n = 0; n < kSlice / 8; ++n) kx[n] = *(const f32x4*)(krow + 8 * n);
    };
#pragma unroll
    for (int n = 0; n < kSlice / 8; ++n) qx[n] = *(const f32x4*)(qrow + 8 * n);
    load_k(0);
    f32x16 acc[kDT];
#pragma unroll
    for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[dt][i] = 0.0f;
    float m = -__builtin_inff(), l = 0.0f;  // l: this lane's half of the keys
#pragma unroll 1
    for (int key0 = 0; key0 < k_seq; key0 += kKeys) {
        f32x16 s;  // element i: key 8 (i / 4) + 4 hf + i % 4
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
        for (int n = 0; n < kSlice / 8; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kx[n][i], qx[n][i], s, 0, 0, 0);
        // the next block's K and this one's V arrive during the exchange
        load_k(key0 + kKeys);
        float vx[16][kDT];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float* vrow = v + (int64_t)min(key0 + 8 * (i >> 2) + 4 * hf + (i & 3), k_seq - 1) * v_stride + col;
#pragma unroll
            for (int dt = 0; dt < kDT; ++dt) vx[i][dt] = vrow[32 * dt];
        }
        __syncthreads();  // the last block's partials are used
#pragma unroll
        for (int u = 0; u < 4; ++u) part[(wave * 4 + u) * 64 + lane] = f32x4{s[4 * u], s[4 * u + 1], s[4 * u + 2], s[4 * u + 3]};
        __syncthreads();
        float mx = -__builtin_inff();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            f32x4 x = part[u * 64 + lane];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) x += part[(w * 4 + u) * 64 + lane];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[4 * u + r] = key0 + 8 * u + 4 * hf + r < k_seq ? x[r] * scale : -__builtin_inff();
                mx = fmaxf(mx, s[4 * u + r]);
            }
        }
        const float m_new = fmaxf(m, fmaxf(mx, __shfl_xor(mx, 32, 64)));
        const float alpha = m == -__builtin_inff() ? 0.0f : expf(m - m_new);
        m = m_new;
        l *= alpha;
#pragma unroll
        for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[dt][i] *= alpha;
        // O^T += V^T P^T; keys that do not exist count as zero rows
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            // -inf weighs nothing, also while there is no finite score; NaN stays
            const float pr = s[i] == -__builtin_inff() ? 0.0f : expf(s[i] - m);
            l += pr;
            const bool in = key0 + 8 * (i >> 2) + 4 * hf + (i & 3) < k_seq;
#pragma unroll
            for (int dt = 0; dt < kDT; ++dt) acc[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? vx[i][dt] : 0.0f, pr, acc[dt], 0, 0, 0);
        }
    }
    const float total = l + __shfl_xor(l, 32, 64);
    const float inv = total != total ? total : 1.0f / fmaxf(total, 1.0e-20f);
    if (col >= rows) return;
    float* row = o + (int64_t)col * o_stride + 4 * hf;
#pragma unroll
    for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
        for (int u = 0; u < 4; ++u)
            *(f32x4*)(row + 32 * dt + 8 * u) = f32x4{acc[dt][4 * u] * inv, acc[dt][4 * u + 1] * inv, acc[dt][4 * u + 2] * inv,
                                                     acc[dt][4 * u + 3] * inv};
}

template <int kN> struct PerLane;
template <> struct PerLane<2> { typedef f32x2 type; };
template <> struct PerLane<4> { typedef f32x4 type; };

template <int kQT, int kDT>
__global__ __launch_bounds__(kWaves * 64, 2) void attention_f32_d512_kernel(OnlineAttentionParams p, int q_blocks) {
    constexpr int kSteps = kSlice / 16;          // K steps of a partial score
    constexpr int kParts = 2 / kDT;              // workgroups that share a query block's output
    constexpr int kRegPlanes = kQT == 2 ? 2 : 3; // Q planes in registers
    constexpr int kPer = 2 * kQT;                // scores per lane of the summed block
    constexpr int kGroup = kKeys / kPer;         // lanes per query there
    constexpr int kPartBytes = kWaves * kQT * 4 * 1024;
    // kQT = 2: the third plane of every K step and the second of the last one
    // (registers that would spill) wait in LDS
    constexpr int kQlBytes = kQT == 2 ? kWaves * kQT * (kSteps + 1) * 1024 : 0;
    constexpr int kProbBytes = kQT * 2 * 3 * 1024;
    __shared__ __attribute__((aligned(16))) char part[kPartBytes];  // [wave][tile][4][64] x 16 bytes
    __shared__ __attribute__((aligned(16))) char qlow[kQlBytes + 16];
    __shared__ __attribute__((aligned(16))) char prob[kProbBytes];  // [tile][16-key half][plane][64] x 16 bytes
    __shared__ float scale_o[32 * kQT];
    __shared__ float total[32 * kQT];
    __shared__ int special, seen[2];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int hf = lane >> 5, col = lane & 31;
    const int task = blockIdx.x / kParts, out_part = blockIdx.x % kParts;
    const int bh = task / q_blocks;
    const int q0 = (task % q_blocks) * (32 * kQT);
    const int h = bh % p.heads, b = bh / p.heads;
    const float* qhead = (const float*)p.q + ((int64_t)b * p.q_seq * p.q_row_stride + (int64_t)h * kDim);
    const float* khead = (const float*)p.k + ((int64_t)b * p.k_seq * p.k_row_stride + (int64_t)h * kDim);
    const float* vhead = (const float*)p.v + ((int64_t)b * p.k_seq * p.v_row_stride + (int64_t)h * kDim);
    float* ohead = (float*)p.o + ((int64_t)b * p.q_seq * p.o_row_stride + (int64_t)h * kDim);
    const char* kslice = (const char*)(khead + kSlice * wave);
    const int out_dim = (kDim / kParts) * out_part + 32 * kDT * wave;  // this wave's first output dim
    const char* vslice = (const char*)(vhead + out_dim);
    const uint32_t k_stride_b = (uint32_t)(p.k_row_stride * 4), v_stride_b = (uint32_t)(p.v_row_stride * 4);
    const int n_blocks = (p.k_seq + kKeys - 1) / kKeys;

    if (threadIdx.x == 0) special = seen[0] = seen[1] = 0;
    __syncthreads();

    // Block t is rows first_row(t) .. +31: a last block that k_seq does not fill
    // starts earlier, at k_seq - 32, and hides the keys that the block before it
    // had, so that every load is of a row that exists (the range check of a
    // load subtracts its scalar offset without a borrow and cannot be relied
    // on). Fewer than 32 keys in all: K rows past the end are caught by that
    // check (their offset is per lane and the scalar one below the size), V by
    // load_v_short.
    auto first_row = [&](int t) __attribute__((always_inline)) { return max(min(t * kKeys, p.k_seq - kKeys), 0); };
    auto block_rows = [&](const char* slice, uint32_t stride_b, int t, int dims) __attribute__((always_inline)) {
        const int rows = min(kKeys, p.k_seq);
        return __builtin_amdgcn_make_buffer_rsrc((void*)(slice + (int64_t)first_row(t) * stride_b), 0,
                                                 (int)((uint32_t)(rows - 1) * stride_b + 4u * dims), 0x00027000);
    };
    // K of block t, K steps 2 half and 2 half + 1: lane holds key col, dims
    // 16 ks + 8 hf .. +7 of the slice.
    f32x4 kraw[kSteps][2];
    const uint32_t k_off = (uint32_t)col * k_stride_b + 32u * hf;
    auto load_k = [&](int t, int half) __attribute__((always_inline)) {
        const auto rows = block_rows(kslice, k_stride_b, t, kSlice);
#pragma unroll
        for (int ks = 2 * half; ks < 2 * half + 2; ++ks)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                kraw[ks][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rows, k_off, 64 * ks + 16 * i, 0));
    };
    // V of 16-key half ss of block t: lane holds keys 16 ss + 8 hf + e, dims
    // kDT col .. + kDT - 1 of the slice.
    float vraw[2][8][kDT];
    const uint32_t v_off = 8u * hf * v_stride_b + 4u * kDT * col;
    auto load_v = [&](int t, int ss) __attribute__((always_inline)) {
        const auto rows = block_rows(vslice, v_stride_b, t, 32 * kDT);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if constexpr (kDT == 2) {
                const f32x2 x = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rows, v_off, (16 * ss + e) * v_stride_b, 0));
                vraw[ss][e][0] = x[0];
                vraw[ss][e][1] = x[1];
            } else {
                vraw[ss][e][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rows, v_off, (16 * ss + e) * v_stride_b, 0));
            }
        }
    };
    auto load_v_short = [&](int ss) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int dt = 0; dt < kDT; ++dt)
                vraw[ss][e][dt] = *(const float*)(vslice + ((uint32_t)min(16 * ss + 8 * hf + e, p.k_seq - 1) * v_stride_b + 4u * (kDT * col + dt)));
    };
    load_k(0, 0);
    load_k(0, 1);

    // Q planes: lane holds query q0 + 32 qt + col, dims 16 ks + 8 hf .. +7.
    i16x8 qop[kQT][kSteps][kRegPlanes];
    const float c = p.scale * 1.4426950408889634f;  // scores to log2 units
    uint32_t q_smallest = ~0u;
    float q_largest = 0.0f;
    char* const qlow_mine = qlow + (kQT == 2 ? wave * kQT * (kSteps + 1) * 1024 : 0) + lane * 16;
#pragma unroll
    for (int qt = 0; qt < kQT; ++qt) {
        const float* row = qhead + (int64_t)min(q0 + 32 * qt + col, p.q_seq - 1) * p.q_row_stride + kSlice * wave + 8 * hf;
#pragma unroll
        for (int ks = 0; ks < kSteps; ++ks) {
            u32x4 pl[3];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x2 x = *(const f32x2*)(row + 16 * ks + 2 * i);
                q_smallest = min(q_smallest, min(nonzero_magnitude(x[0]), nonzero_magnitude(x[1])));
                q_largest = fmaxf(q_largest, fmaxf(fabsf(x[0]), fabsf(x[1])));
                uint32_t w[3];
                split2<3, false>(x[0], x[1], w);
#pragma unroll
                for (int j = 0; j < 3; ++j) pl[j][i] = w[j];
            }
#pragma unroll
            for (int j = 0; j < kRegPlanes; ++j) qop[qt][ks][j] = __builtin_bit_cast(i16x8, pl[j]);
            if constexpr (kQT == 2) {
                *(lds_u32x4*)(qlow_mine + (qt * (kSteps + 1) + ks) * 1024) = pl[2];
                if (ks == kSteps - 1) *(lds_u32x4*)(qlow_mine + (qt * (kSteps + 1) + kSteps) * 1024) = pl[1];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    if (!planes_carry_queries(q_smallest, q_largest, c)) special = 1;

    f32x16 o[kQT][kDT];  // [tile][dt]: dims kDT m + dt of the slice, m the tile row
#pragma unroll
    for (int qt = 0; qt < kQT; ++qt)
#pragma unroll
        for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[qt][dt][i] = 0.0f;

    // Planes of the next matrix operand, formed while the matrix cores work on
    // the current one (two sets in turn).
    struct Operand { i16x8 pl[3]; };
    auto split8 = [&](const float (&x)[8]) __attribute__((always_inline)) {
        u32x4 pl[3];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t w[3];
            split2<3, false>(x[2 * i], x[2 * i + 1], w);
#pragma unroll
            for (int j = 0; j < 3; ++j) pl[j][i] = w[j];
        }
        return Operand{{__builtin_bit_cast(i16x8, pl[0]), __builtin_bit_cast(i16x8, pl[1]), __builtin_bit_cast(i16x8, pl[2])}};
    };
    auto split_k = [&](int ks) __attribute__((always_inline)) {
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = kraw[ks][i >> 2][i & 3];
        return split8(x);
    };
    auto split_v = [&](int ss, int dt) __attribute__((always_inline)) {
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = vraw[ss][i][dt];
        return split8(x);
    };
    // partial scores, K step ks
    f32x16 s[kQT];
    i16x8 qlo[kQT];  // third plane of Q, read from LDS a stage ahead
    auto read_qlow = [&](int ks) __attribute__((always_inline)) {
        if constexpr (kQT == 2)
#pragma unroll
            for (int qt = 0; qt < kQT; ++qt) qlo[qt] = __builtin_bit_cast(i16x8, *(const lds_u32x4*)(qlow_mine + (qt * (kSteps + 1) + ks) * 1024));
    };
    auto scores_step = [&](int ks, const Operand& k, const i16x8 (&low)[kQT]) __attribute__((always_inline)) {
#pragma unroll
        for (int qt = 0; qt < kQT; ++qt) {
            i16x8 ql;
            if constexpr (kQT == 2) ql = low[qt];
            else ql = qop[qt][ks][2];
            i16x8 qm = qop[qt][ks][1];
            if constexpr (kQT == 2)
                if (ks == kSteps - 1) qm = __builtin_bit_cast(i16x8, *(const lds_u32x4*)(qlow_mine + (qt * (kSteps + 1) + kSteps) * 1024));
            s[qt] = mfma32<false>(k.pl[2], qop[qt][ks][0], s[qt]);
            s[qt] = mfma32<false>(k.pl[1], qm, s[qt]);
            s[qt] = mfma32<false>(k.pl[1], qop[qt][ks][0], s[qt]);
            s[qt] = mfma32<false>(k.pl[0], ql, s[qt]);
            s[qt] = mfma32<false>(k.pl[0], qm, s[qt]);
            s[qt] = mfma32<false>(k.pl[0], qop[qt][ks][0], s[qt]);
        }
    };
    // O^T of dims dt += V^T P^T over a 16-key half
    struct Probs { i16x8 pl[kQT][3]; };
    auto read_probs = [&](int ss) __attribute__((always_inline)) {
        Probs r;
#pragma unroll
        for (int qt = 0; qt < kQT; ++qt)
#pragma unroll
            for (int pl = 0; pl < 3; ++pl)
                r.pl[qt][pl] = __builtin_bit_cast(i16x8, *(const lds_u32x4*)(prob + ((qt * 2 + ss) * 3 + pl) * 1024 + lane * 16));
        return r;
    };
    auto output_step = [&](int dt, const Operand& v, const Probs& probs) __attribute__((always_inline)) {
#pragma unroll
        for (int qt = 0; qt < kQT; ++qt) {
            const i16x8 (&pop)[3] = probs.pl[qt];
            o[qt][dt] = mfma32<false>(v.pl[2], pop[0], o[qt][dt]);
            o[qt][dt] = mfma32<false>(v.pl[1], pop[1], o[qt][dt]);
            o[qt][dt] = mfma32<false>(v.pl[0], pop[2], o[qt][dt]);
            o[qt][dt] = mfma32<false>(v.pl[1], pop[0], o[qt][dt]);
            o[qt][dt] = mfma32<false>(v.pl[0], pop[1], o[qt][dt]);
            o[qt][dt] = mfma32<false>(v.pl[0], pop[0], o[qt][dt]);
        }
    };
    // Ends a stage: its matrix instructions spread over its other work, kValu
    // vector instructions after each.
    auto stage_end = [&]<int kValu>() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 6 * kQT; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);  // VALU
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto clear_scores = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int qt = 0; qt < kQT; ++qt)
#pragma unroll
            for (int i = 0; i < 16; ++i) s[qt][i] = 0.0f;
    };
    // Partials: element 4u + r is key 8u + 4hf + r of query col; 16-byte unit
    // (hf, col) of [tile][u] sits at column col ^ 2 (2u + hf), so that the
    // summing lanes (8 units of one column each) reach distinct banks.
    auto write_partials = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int qt = 0; qt < kQT; ++qt)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                char* dst = part + ((wave * kQT + qt) * 4 + u) * 1024 + (32 * hf + (col ^ (2 * (2 * u + hf)))) * 16;
                *(lds_f32x4*)dst = f32x4{s[qt][4 * u], s[qt][4 * u + 1], s[qt][4 * u + 2], s[qt][4 * u + 3]};
            }
    };

    // This lane's share of the summed scores: query sq of tile st, keys
    // 8 su + 4 sh + sr .. + kPer - 1.
    const int j = lane % kGroup;
    const int st = kQT == 2 ? wave >> 2 : 0;
    const int sq = (64 / kGroup) * (kQT == 2 ? wave & 3 : wave) + lane / kGroup;
    const int su = kQT == 2 ? j >> 1 : j >> 2, sh = kQT == 2 ? j & 1 : (j >> 1) & 1, sr = kQT == 2 ? 0 : 2 * (j & 1);
    const char* const part_mine = part + (st * 4 + su) * 1024 + (32 * sh + (sq ^ (2 * (2 * su + sh)))) * 16 + 4 * sr;
    // B operand of P.V: 16-key half ss, lane (hf', query): keys 16 ss + 8 hf' + e
    char* const prob_mine = prob + (st * 2 + (su >> 1)) * 3 * 1024 + (32 * (su & 1) + sq) * 16 + 8 * sh + 2 * sr;
    float m_run = -__builtin_inff(), l_run = 0.0f;  // of query sq; this lane's part of the sum

    float sc[kPer];
    typedef typename PerLane<kPer>::type part_t;
    part_t parts[kWaves / 2];
    auto read_partials = [&](int half) __attribute__((always_inline)) {
#pragma unroll
        for (int w = 0; w < kWaves / 2; ++w)
            parts[w] = *(const __attribute__((address_space(3))) part_t*)(part_mine + (half * (kWaves / 2) + w) * (kQT * 4 * 1024));
    };
    auto sum_partials = [&](int half) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const float x = (parts[0][i] + parts[1][i]) + (parts[2][i] + parts[3][i]);
            sc[i] = half == 0 ? x : sc[i] + x;
        }
    };
    auto softmax = [&]<bool kLast>(int t) __attribute__((always_inline)) {
        if constexpr (kLast) {
            // visible: keys of the last block from t kKeys on, below k_seq
            const int before = t * kKeys - first_row(t), n = min(p.k_seq, kKeys);
            const int mine = 8 * su + 4 * sh + sr;
#pragma unroll
            for (int i = 0; i < kPer; ++i) sc[i] = mine + i >= before && mine + i < n ? sc[i] : -__builtin_inff();
        }
        float mx = sc[0];
#pragma unroll
        for (int i = 1; i < kPer; ++i) mx = fmaxf(mx, sc[i]);
        mx = group_max<kGroup>(mx) * c;
        const float m_new = fmaxf(m_run, mx);  // finite: every block holds a visible key
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);  // 0 on the first block
        m_run = m_new;
        float pr[kPer], sum = 0.0f;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            pr[i] = 65536.0f * __builtin_amdgcn_exp2f(__builtin_fmaf(sc[i], c, -m_new));  // small ones keep their planes
            sum += pr[i];
        }
        l_run = l_run * alpha + sum;
        uint32_t w[kPer / 2][3];
#pragma unroll
        for (int i = 0; i < kPer / 2; ++i) split2<3, false>(pr[2 * i], pr[2 * i + 1], w[i]);
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) {
            if constexpr (kQT == 2) *(lds_u32x2*)(prob_mine + pl * 1024) = u32x2{w[0][pl], w[1][pl]};
            else *(lds_u32*)(prob_mine + pl * 1024) = w[0][pl];
        }
        if (j == 0) scale_o[32 * st + sq] = alpha;
    };

    clear_scores();
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks) {
        read_qlow(ks);
        scores_step(ks, split_k(ks), qlo);
        __builtin_amdgcn_sched_barrier(0);
    }
    write_partials();
    read_qlow(0);
    Operand even = {}, odd = {};
    if constexpr (kQT == 1) {
        if (p.k_seq < kKeys) {
            load_v_short(0);
            load_v_short(1);
        } else {
            load_v(0, 0);
            load_v(0, 1);
        }
    }
    if (n_blocks > 1) {
        load_k(1, 0);
        load_k(1, 1);
        even = split_k(0);
    }
    auto rescale = [&]() __attribute__((always_inline)) {
        float alpha[kQT];
        bool move = false;
#pragma unroll
        for (int qt = 0; qt < kQT; ++qt) {
            alpha[qt] = scale_o[32 * qt + col];
            move = move || alpha[qt] != 1.0f;
        }
        if (__builtin_amdgcn_ballot_w64(move) != 0) {
#pragma unroll
            for (int qt = 0; qt < kQT; ++qt)
#pragma unroll
                for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[qt][dt][i] *= alpha[qt];
        }
    };

    // Block t: scores of t + 1, output of t (the last block has no next one).
    constexpr int kFill = 8 / kQT;  // vector instructions per matrix instruction
    auto scores_stage = [&]<int kStep>(const Operand& now, auto&& other) __attribute__((always_inline)) {
        i16x8 low[kQT];
#pragma unroll
        for (int qt = 0; qt < kQT; ++qt) low[qt] = qlo[qt];
        if constexpr (kStep + 1 < kSteps) read_qlow(kStep + 1);
        other();
        scores_step(kStep, now, low);
        stage_end.template operator()<kStep == 2 ? 2 * kFill : kFill>();
    };
    for (int t = 0; t + 1 < n_blocks; ++t) {
        // Loads: kQT = 1 a block ahead; kQT = 2, whose registers are full, two
        // or three stages ahead, into what the last operands left. K of the
        // block after next past the end: of the last block, unused.
        const int t2 = min(t + 2, n_blocks - 1);
        __syncthreads();  // partials of t there; probabilities of t - 1 used
        clear_scores();
        read_partials(0);
        scores_stage.template operator()<0>(even, [&]() __attribute__((always_inline)) { odd = split_k(1); });
        if constexpr (kQT == 2) load_v(t, 0);
        else load_k(t2, 0);
        sum_partials(0);
        read_partials(1);
        scores_stage.template operator()<1>(odd, [&]() __attribute__((always_inline)) { even = split_k(2); });
        sum_partials(1);
        scores_stage.template operator()<2>(even, [&]() __attribute__((always_inline)) {
            odd = split_k(3);
            softmax.template operator()<false>(t);
        });
        if constexpr (kQT == 2) load_v(t, 1);
        else load_k(t2, 1);
        scores_stage.template operator()<3>(odd, [&]() __attribute__((always_inline)) { even = split_v(0, 0); });
        __syncthreads();  // probabilities of t there; partials of t used
        Probs first = read_probs(0);
        rescale();
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kQT == 2) load_k(t2, 0);
        odd = split_v(kDT == 2 ? 0 : 1, kDT - 1);
        output_step(0, even, first);
        write_partials();
        stage_end.template operator()<kFill>();
        if constexpr (kQT == 1) load_v(t + 1, 0);
        Probs second = read_probs(1);
        if constexpr (kDT == 2) {
            even = split_v(1, 0);
            output_step(1, odd, first);
            stage_end.template operator()<kFill>();
            if constexpr (kQT == 2) load_k(t2, 1);
            odd = split_v(1, 1);
            output_step(0, even, second);
            stage_end.template operator()<kFill>();
        }
        if constexpr (kQT == 1) load_v(t + 1, 1);
        read_qlow(0);
        even = split_k(0);
        output_step(kDT - 1, odd, second);
        stage_end.template operator()<kFill>();
    }
    __syncthreads();
    if constexpr (kQT == 2) {
        load_v(n_blocks - 1, 0);
        load_v(n_blocks - 1, 1);
    }
    read_partials(0);
    sum_partials(0);
    read_partials(1);
    sum_partials(1);
    softmax.template operator()<true>(n_blocks - 1);
    __syncthreads();
    rescale();
#pragma unroll
    for (int ss = 0; ss < 2; ++ss)
#pragma unroll
        for (int dt = 0; dt < kDT; ++dt) {
            output_step(dt, split_v(ss, dt), read_probs(ss));
            __builtin_amdgcn_sched_barrier(0);
        }

    l_run = group_sum<kGroup>(l_run);
    if (j == 0) total[32 * st + sq] = l_run;
    __syncthreads();
    // Planes turn an infinity, a NaN or an FP32 value above the largest bf16
    // into a NaN, which reaches every score or output that it meets: such
    // workgroups (and those whose results overflow, or are so small that planes
    // may have lost bits of them) start over in fp32, unless a NaN has decided
    // all of their results.
    float bad = 0.0f;
    uint32_t smallest = ~0u;
#pragma unroll
    for (int qt = 0; qt < kQT; ++qt) {
        const float inv = 1.0f / fmaxf(total[32 * qt + col], 1.0e-20f);
#pragma unroll
        for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                o[qt][dt][i] *= inv;
                bad = __builtin_fmaf(o[qt][dt][i], 0.0f, bad);
                smallest = min(smallest, nonzero_magnitude(o[qt][dt][i]));
            }
    }
    if (results_too_small(smallest) || bad != bad) special = 1;
    __syncthreads();
    bool redo = __builtin_amdgcn_readfirstlane(special) != 0;
    if (__builtin_expect(redo, 0))
        redo = !all_rows_nan(qhead + (int64_t)q0 * p.q_row_stride, khead, p.q_row_stride, p.k_row_stride, min(32 * kQT, p.q_seq - q0),
                             p.k_seq, (__attribute__((address_space(3))) int*)seen);
    if (__builtin_expect(redo, 0)) {
#pragma unroll 1
        for (int first = q0; first < min(q0 + 32 * kQT, p.q_seq); first += 32)
            redo_block<kDT>(qhead + (int64_t)first * p.q_row_stride, khead, vhead + out_dim, ohead + (int64_t)first * p.o_row_stride + out_dim,
                            p.q_row_stride, p.k_row_stride, p.v_row_stride, p.o_row_stride, min(32, p.q_seq - first), p.k_seq, p.scale,
                            (lds_f32x4*)part);
        return;
    }
    // lane holds tile rows m = 8u + 4hf + r of query col: dims kDT m + dt
#pragma unroll
    for (int qt = 0; qt < kQT; ++qt) {
        const int query = q0 + 32 * qt + col;
        if (query >= p.q_seq) continue;
        float* row = ohead + (int64_t)query * p.o_row_stride + out_dim + 4 * kDT * hf;
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int n = 0; n < 4 * kDT; n += 4) {
                f32x4 w;
#pragma unroll
                for (int i = 0; i < 4; ++i) w[i] = o[qt][(n + i) % kDT][4 * u + (n + i) / kDT];
                *(f32x4*)(row + 8 * kDT * u + n) = w;
            }
    }
}

}  // namespace

bool attention_f32_d512_eligible(const OnlineAttentionParams& p, int dtype) {
    auto a16 = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
    return dtype == 2 && p.head_dim == kDim && !p.causal && p.key_mask == nullptr && p.k_seq > 0 &&
           p.q_row_stride % 4 == 0 && p.k_row_stride % 4 == 0 && p.v_row_stride % 4 == 0 && p.o_row_stride % 4 == 0 &&
           a16(p.q) && a16(p.k) && a16(p.v) && a16(p.o) &&
           (int64_t)kKeys * p.k_row_stride * 4 < (int64_t{1} << 31) && (int64_t)kKeys * p.v_row_stride * 4 < (int64_t{1} << 31);
}

hipError_t launch_attention_f32_d512(const OnlineAttentionParams& p, int compute_units, hipStream_t stream) {
    if (p.batch == 0 || p.q_seq == 0) return hipSuccess;
    // One workgroup per CU at a time. 64 queries per workgroup take 1.65x the
    // time of 32 per key block (16384 tokens: 2.6 ms against 3.1 in two rounds
    // of 32); with at most half the CUs' worth of 32-query blocks, two
    // workgroups share a block's output dims (each forms all of its scores).
    const int64_t heads_total = (int64_t)p.heads * p.batch;
    const int64_t cus = compute_units > 0 ? compute_units : 256;
    const int64_t b64 = ((int64_t)p.q_seq + 63) / 64, b32 = ((int64_t)p.q_seq + 31) / 32;
    const int64_t r64 = (b64 * heads_total + cus - 1) / cus, r32 = (b32 * heads_total + cus - 1) / cus;
    const bool wide = 5 * r64 <= 3 * r32 && p.k_seq >= kKeys;  // 64 queries: no short last block
    const int64_t grid = (wide ? b64 : 2 * b32 * heads_total <= cus ? 2 * b32 : b32) * heads_total;
    if (grid > INT32_MAX) return hipErrorInvalidValue;
    const dim3 g((unsigned)grid), block(kWaves * 64);
    if (wide) hipLaunchKernelGGL((attention_f32_d512_kernel<2, 2>), g, block, 0, stream, p, (int)b64);
    else if (2 * b32 * heads_total <= cus) hipLaunchKernelGGL((attention_f32_d512_kernel<1, 1>), g, block, 0, stream, p, (int)b32);
    else hipLaunchKernelGGL((attention_f32_d512_kernel<1, 2>), g, block, 0, stream, p, (int)b32);
    return hipGetLastError();
}

}  // namespace sdxl_hip
