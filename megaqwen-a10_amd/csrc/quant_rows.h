// The weight quantizers' row pass, shared by the three formats (quant.hip, formats.hip):
//   INT8  s = bf16(amax / 127) per row,          q = clamp(rint(w / s), -128, 127), one byte
//   FP8   s = fp32(amax / 448) per row,          q = E4M3 code of w / s, one byte
//   INT4  s = bf16(amax / 7) per 128 elements,   q = clamp(rint(w / s), -8, 7), a nibble
// s widened to fp32 and at least 1e-12, IEEE divisions, ties to even.
//
// Bound by memory: 2 bytes in and 1 (INT4: 0.53) out per element. A wave takes a row at a time, its
// elements in registers from one 16-byte load per lane and 512 elements, so the row is read
// once, and requests its next row before it works on this one; a grid of at most 8 workgroups
// per CU strides over the rows (a workgroup per row of 2-byte loads, read twice, spent its
// time on launching workgroups and issuing loads). [151936, 1024]: INT8 285 -> 84-88 us (5.3-5.6 TB/s,
// what a copy reaches), FP8 297 -> 101-107, INT4 (a thread per group) 767 -> 81-89.
// The per-element division is three multiply-adds: with r = RN(1 / s), q = RN(w r) and the
// remainder w - q s, RN(q + remainder r) is the correctly rounded w / s (P. Markstein,
// "Computation of elementary functions on the IBM RISC System/6000 processor", IBM J. Res.
// Dev. 34, 1990; his q is within one unit of w / s and the remainder exact, here q can be half a
// unit further off, and every pair of mantissas that w and s can have was checked). It needs s
// finite (else the IEEE division is used); where w is so small that the remainder underflows, w / s
// is below 2^-60 either way and its code is 0.
#pragma once

#include "common.h"

namespace mq {

enum QuantFormat { Q_INT8 = 0, Q_FP8 = 1, Q_INT4 = 2 };
constexpr int kQRowThreads = 256;
constexpr int kQRowWaves = kQRowThreads / kWave;
constexpr int kQRowChunk = 8 * kWave;             // elements of one 16-byte load per lane
constexpr int kQRowMaxChunks = 16;                // longest row held in registers: 8192 elements

__device__ __forceinline__ uint32_t fp8_e4m3_encode(float x) {
    const uint32_t sign = (__float_as_uint(x) >> 24) & 0x80u;
    const float a = fabsf(x);
    if (!(a < 448.0f)) return sign | 0x7Eu;                       // saturate (and NaN)
    if (a < 0x1p-6f) return sign | (uint32_t)__builtin_rintf(a * 512.0f);   // subnormal: m 2^-9, exact scaling
    const uint32_t u = __float_as_uint(a);
    const uint32_t r = (u + 0x7FFFFu + ((u >> 20) & 1u)) & 0xFFF00000u;      // mantissa to 3 bits, RNE
    const int e = (int)(r >> 23) - 127;
    return sign | ((uint32_t)(e + 7) << 3) | ((r >> 20) & 7u);
}

// w / s for s > 0, with w's sign also on a zero; kFast: s finite, r = RN(1 / s)
template <bool kFast>
__device__ __forceinline__ float quant_div(float w, float s, float r) {
    if constexpr (!kFast) return __fdiv_rn(w, s);
    const float q = w * r;
    return copysignf(fmaf(fmaf(-q, s, w), r, q), w);
}

template <int F>
__device__ __forceinline__ float quant_scale(float amax) {
    if constexpr (F == Q_FP8) return fmaxf(__fdiv_rn(amax, 448.0f), 1e-12f);
    else return fmaxf(round_bf16(__fdiv_rn(amax, F == Q_INT8 ? 127.0f : 7.0f)), 1e-12f);
}

template <int F>
__device__ __forceinline__ uint32_t quant_code(float v) {
    if constexpr (F == Q_FP8) return fp8_e4m3_encode(v);
    else if constexpr (F == Q_INT8) return (uint32_t)(int)fminf(fmaxf(__builtin_rintf(v), -128.0f), 127.0f) & 0xffu;
    else return (uint32_t)(int)fminf(fmaxf(__builtin_rintf(v), -8.0f), 7.0f) & 15u;
}

// Rows of at most 512 C elements, K % 8 == 0 (INT4: K % 128 == 0), 16-byte aligned w, q aligned
// to a lane's 8 codes.
template <int F, int C>
__global__ void __launch_bounds__(kQRowThreads)
quantize_rows_wave_kernel(const uint16_t* __restrict__ w, int M, int K, uint8_t* __restrict__ q, float* __restrict__ scale) {
    const int lane = threadIdx.x % kWave;
    const uint32_t stride = gridDim.x * kQRowWaves;       // M + stride < 2^32
    uint32_t row = blockIdx.x * kQRowWaves + threadIdx.x / kWave;
    uint4 next[C];
    auto load = [&](uint32_t r) {
        const uint16_t* const wr = w + (int64_t)r * K + 8 * lane;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            next[c] = make_uint4(0, 0, 0, 0);               // elements past the row: zero
            if (c * kQRowChunk + 8 * lane < K) next[c] = ldg16_stream(wr + c * kQRowChunk);
        }
    };
    if (row < (uint32_t)M) load(row);
    for (; row < (uint32_t)M; row += stride) {
        uint4 v[C];
#pragma unroll
        for (int c = 0; c < C; ++c) v[c] = next[c];
        if (row + stride < (uint32_t)M) load(row + stride);
        auto elem = [&](int c, int i) {
            const uint32_t u = i < 2 ? v[c].x : i < 4 ? v[c].y : i < 6 ? v[c].z : v[c].w;
            return __uint_as_float((i & 1) ? u & 0xffff0000u : u << 16);
        };
        float m[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            m[c] = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) m[c] = fmaxf(m[c], fabsf(elem(c, i)));
        }
        float s = 0.0f, r = 0.0f;
        bool ok = true;
        if constexpr (F != Q_INT4) {
#pragma unroll
            for (int c = 1; c < C; ++c) m[0] = fmaxf(m[0], m[c]);
            s = quant_scale<F>(wave_max(m[0]));
            r = __fdiv_rn(1.0f, s);
            ok = s < INFINITY;
            if (lane == 0) scale[row] = s;
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            if (c * kQRowChunk >= K) break;                 // uniform
            const int k = c * kQRowChunk + 8 * lane;
            if constexpr (F == Q_INT4) {
                float g = m[c];                             // a group: the 16 lanes of a DPP row
                g = fmaxf(g, partner<1>(g));
                g = fmaxf(g, partner<2>(g));
                g = fmaxf(g, partner<4>(g));
                g = fmaxf(g, partner<8>(g));
                s = quant_scale<F>(g);
                r = __fdiv_rn(1.0f, s);
                ok = s < INFINITY;
                if ((lane & 15) == 0 && k < K) scale[(int64_t)row * (K / 128) + k / 128] = s;
            }
            uint32_t code[8];
            if (__all(ok)) {
#pragma unroll
                for (int i = 0; i < 8; ++i) code[i] = quant_code<F>(quant_div<true>(elem(c, i), s, r));
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) code[i] = quant_code<F>(quant_div<false>(elem(c, i), s, r));
            }
            if (k < K) {
                if constexpr (F == Q_INT4) {
                    uint32_t out = 0;
#pragma unroll
                    for (int i = 0; i < 8; ++i) out |= code[i] << (4 * i);
                    *reinterpret_cast<uint32_t*>(q + (int64_t)row * (K / 2) + k / 2) = out;
                } else {
                    *reinterpret_cast<uint2*>(q + (int64_t)row * K + k) =
                        make_uint2(code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24),
                                   code[4] | (code[5] << 8) | (code[6] << 16) | (code[7] << 24));
                }
            }
        }
    }
}

// Whether the row pass takes these rows: whole lanes of 8 elements, at most 8192 of them, and
// pointers aligned to a lane's load and store. The other rows go through the formats' element
// kernels (and FP8 matrices of few rows, launch_quantize_fp8).
inline bool quant_rows_fit(const void* w, int K, const void* q, int code_bytes) {
    return K % 8 == 0 && K <= kQRowMaxChunks * kQRowChunk && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(q) % code_bytes == 0;
}

template <int F>
void launch_quant_rows(const void* w, int M, int K, uint8_t* q, float* scale, int cus, hipStream_t stream) {
    const int want = (M - 1) / kQRowWaves + 1;
    const dim3 grid(want < 8 * cus ? want : 8 * cus), block(kQRowThreads);
    const uint16_t* const wb = static_cast<const uint16_t*>(w);
    const int C = (K + kQRowChunk - 1) / kQRowChunk;
    if (C <= 2) hipLaunchKernelGGL((quantize_rows_wave_kernel<F, 2>), grid, block, 0, stream, wb, M, K, q, scale);
    else if (C <= 4) hipLaunchKernelGGL((quantize_rows_wave_kernel<F, 4>), grid, block, 0, stream, wb, M, K, q, scale);
    else if (C <= 8) hipLaunchKernelGGL((quantize_rows_wave_kernel<F, 8>), grid, block, 0, stream, wb, M, K, q, scale);
    else hipLaunchKernelGGL((quantize_rows_wave_kernel<F, 16>), grid, block, 0, stream, wb, M, K, q, scale);
}

}  // namespace mq
