// Weight-only matvec of one-byte weights with per-row scales, y[j] = scale[j] * sum_k x[k] *
// w[j,k] (INT8: gemv.hip, FP8: formats.hip), fp32 activations and sums.
//
// Layout: one 64-lane wave owns R consecutive rows at a time; each lane reads 16 contiguous
// weights of a row per 1 KB chunk (a coalesced 1 KB row segment per wave instruction) and has
// the activations of its own 16 columns of every chunk in registers for all its rows. The R row
// sums are finished with a transpose reduction (R values -> 1 per lane group).
//
// Bound by memory: HBM for large matrices, and for a few MB one memory round trip, so a wave
// requests its first rows before anything else, the activations (L2 after the first wave) right
// behind them, and each further item's rows while it computes the one before. No LDS and no
// workgroup barrier. (The activations staged through LDS by the workgroup, element by element,
// before the first weight load: kernel times on matrices read in turn [2048, 6144] 7.9 us against
// 7.7 now, [1024, 3072] 4.4 / 3.6, [1024, 2048] 3.7 / 3.2, [151936, 1024] 32.8 / 28.6.)
// R is the largest for the row length (R rows x chunks of 16 bytes per lane in flight) that
// still gives every CU two workgroups of items, so that small shapes spread over every CU.
//
// Rows past 8192 elements: activations in registers would leave one wave per SIMD (436 registers at
// 16 chunks), so the workgroup stages them in LDS, 16 bytes per load, behind its waves' first
// weights. [4096, 9216] 23.8 -> 11.4 us, [4096, 12288] 28.7 -> 14.1, [16384, 16384] 69.8 -> 51.4.
// Rows shorter than a chunk: a row leaves lanes idle and a wave has fewer bytes in flight, so there
// are eight workgroups a CU, with the registers of the next item's rows given up for it.
// [100000, 256] 14.7 -> 12.2 us, [100000, 640] 17.8 -> 15.0, [65536, 768] 13.0 -> 11.4.
//
// The weights are streamed past the caches, where the next matrix of a model would displace them
// anyway ([151936, 1024] 32.2 -> 28.7 us a call), but for matrices of 8 to 32 MB: these may still be in the
// L2s (8 x 4 MB) from the call before and take much longer from memory. Kernel us, streamed / not:
// called again and again [12288, 2048] 6.9 / 4.9, [2048, 6144] 6.4 / 5.6, [32768, 1024] 7.4 / 6.3; read in turn
// with others, past every cache, 7.6 / 8.3, 7.0 / 7.6, 8.5 / 9.3. Up to 8 MB a call is one memory round trip,
// shorter than its host time: [6144, 1024] again 3.4 / 3.0, in turn 3.7 / 4.2; [4096, 1024] 2.9 / 2.8 and
// 3.4 / 3.5. Past 32 MB: [49152, 1024] 10.7 / 11.5 and 12.0 / 12.9.
//
// Repeat mode (steady-state measurement): one launch computes `reps` matvecs, rep i against
// weight copy i % n_copies (copies `copy_stride` bytes apart, output row block i % n_copies of
// y). The items (rep, row batch) are independent, so the waves stream weights without a launch
// or a ramp between matvecs; reps = n_copies = 1 is the plain call.
#pragma once

#include <algorithm>

#include "common.h"
#include "internal.h"

namespace mq {

constexpr int kGemvThreads = 256;
constexpr int kGemvWaves = kGemvThreads / kWave;
constexpr int64_t kGemvCachedMin = 8 << 20, kGemvCachedMax = 32 << 20;     // bytes of weights not streamed

// Activations in LDS (rows past 8192 elements)
constexpr bool gemv_lds(int chmax) { return chmax > 8; }
// Workgroups per CU: LM head [151936, 1024] 2 32.4 us, 4 28.0, 8 28.6; with the activations in LDS as many
// as fit ([16384, 16384] 2 50.8 us, 3 58.5); without a next item's rows 8
constexpr int gemv_per_cu(int chmax, bool ahead) { return !ahead ? 8 : !gemv_lds(chmax) ? 4 : chmax <= 12 ? 3 : 2; }

// F::dot(w, x, acc): 16 weights against x[0..3], the activations of elements 4 i .. 4 i + 3.
// kStream: loads past the caches; kAhead: an item's rows are requested before the one before it is
// computed.
template <class F, int R, int CHMAX, bool kStream, bool kAhead>
__global__ void __launch_bounds__(kGemvThreads)
gemv_rows_kernel(const float* __restrict__ x, const uint8_t* __restrict__ w, int64_t copy_stride, int n_copies,
                 const float* __restrict__ scale, float* __restrict__ y, int M, int K, int reps) {
    constexpr bool kLds = gemv_lds(CHMAX);
    extern __shared__ float4 xs[];
    const int lane = threadIdx.x % kWave;
    const uint32_t total_waves = gridDim.x * kGemvWaves;
    const uint32_t nbatch = (M + R - 1) / R;
    const uint32_t items = (uint32_t)reps * nbatch;         // < 2^31: reps M is (checked by the host)
    uint32_t it = blockIdx.x * kGemvWaves + threadIdx.x / kWave;
    uint4 next[R][CHMAX];
    auto load = [&](uint32_t i) {
        const uint32_t rep = reps > 1 ? i / nbatch : 0;
        const int row0 = (int)(i - rep * nbatch) * R;
        const uint8_t* const wc = w + (int64_t)(rep % (uint32_t)n_copies) * copy_stride;
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < CHMAX; ++c) {
                next[r][c] = make_uint4(0, 0, 0, 0);
                const int col = c * 1024 + lane * 16;
                if (row0 + r < M && col < K)
                    next[r][c] = (kStream ? ldg16_stream : ldg16)(wc + (int64_t)(row0 + r) * K + col);
            }
    };
    if (it < items) load(it);
    float4 xv[kLds ? 1 : CHMAX][4];
    if constexpr (kLds) {
        // piece i of a lane's 16 activations of chunk c at xs[64 (4 c + i) + lane]
        for (int f = threadIdx.x; f < (K + 1023) / 1024 * 256; f += kGemvThreads)
            xs[(f / 256 * 4 + f % 4) * kWave + f % 256 / 4] =
                4 * f < K ? reinterpret_cast<const float4*>(x)[f] : make_float4(0.f, 0.f, 0.f, 0.f);
        __syncthreads();
    } else {
#pragma unroll
        for (int c = 0; c < CHMAX; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int col = c * 1024 + lane * 16;
                xv[c][i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (col < K) xv[c][i] = reinterpret_cast<const float4*>(x + col)[i];
            }
    }
    for (; it < items; it += total_waves) {
        uint4 wv[R][CHMAX];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < CHMAX; ++c) wv[r][c] = next[r][c];
        if (kAhead && it + total_waves < items) load(it + total_waves);
        float acc[R];
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = 0.0f;
#pragma unroll
        for (int c = 0; c < CHMAX; ++c) {
            if (CHMAX <= 4 || c * 1024 < K) {               // uniform: no work for chunks past the row
                if constexpr (kLds) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) xv[0][i] = xs[(4 * c + i) * kWave + lane];
                }
#pragma unroll
                for (int r = 0; r < R; ++r) acc[r] = F::dot(wv[r][c], xv[kLds ? 0 : c], acc[r]);
            }
        }
        const float s = transpose_reduce<R>(acc, lane);
        constexpr int span = kWave / R;
        const uint32_t rep = reps > 1 ? it / nbatch : 0;
        const int row = (int)(it - rep * nbatch) * R + lane / span;
        if ((lane % span) == 0 && row < M) y[(int64_t)(rep % (uint32_t)n_copies) * M + row] = s * scale[row];
        if (!kAhead && it + total_waves < items) load(it + total_waves);
    }
}

template <class F, int R, int CHMAX, bool kAhead>
int launch_gemv_rows_t(const float* x, const uint8_t* w, int64_t copy_stride, int n_copies, const float* scale, float* y,
                       int M, int K, int reps, hipStream_t stream) {
    const int64_t items = (int64_t)reps * ((M + R - 1) / R);
    // at most gemv_per_cu workgroups a CU, and no more waves than give each the same number of items,
    // in whole workgroups per CU: [151936, 1024] with 950 workgroups on 256 CUs took 28.0 us a call (INT8)
    // and 27.4 (FP8), with 1024 27.2 and 26.6 (three alternating runs, spread 0.15 at most)
    const int64_t cus = device_cu_count();
    const int64_t most = gemv_per_cu(CHMAX, kAhead) * cus * kGemvWaves;
    const int64_t per = (items + most - 1) / most;
    const int64_t waves = (items + per - 1) / per;
    const int64_t even = (waves + kGemvWaves - 1) / kGemvWaves;
    const int grid = (int)(per > 1 ? (even + cus - 1) / cus * cus : even);
    const size_t lds = gemv_lds(CHMAX) ? (size_t)(K + 1023) / 1024 * 4096 : 0;          // at most 64 KB
    const bool cached = (int64_t)M * K > kGemvCachedMin / n_copies && (int64_t)M * K <= kGemvCachedMax / n_copies;
    hipLaunchKernelGGL((cached ? gemv_rows_kernel<F, R, CHMAX, false, kAhead> : gemv_rows_kernel<F, R, CHMAX, true, kAhead>),
                       dim3(grid), dim3(kGemvThreads), lds, stream, x, w, copy_stride, n_copies, scale, y, M, K, reps);
    return check_launch("gemv_rows_kernel");
}

template <class F>
int launch_gemv_rows(const float* x, const uint8_t* w, int64_t copy_stride, int n_copies, const float* scale, float* y,
                     int M, int K, int reps, hipStream_t stream) {
    const int CH = (K + 1023) / 1024;
    int R = CH <= 1 ? 8 : CH == 2 ? 4 : CH <= 4 ? 2 : 1;
    const int64_t min_waves = (int64_t)2 * kGemvWaves * device_cu_count();
    while (R > 1 && (int64_t)reps * ((M + R - 1) / R) < min_waves) R /= 2;
#define MQ_GEMV(RR, CC, AHEAD)                                                                                     \
    if (CH <= CC && R == RR) return launch_gemv_rows_t<F, RR, CC, AHEAD>(x, w, copy_stride, n_copies, scale, y, M, K, reps, stream)
    if (K < 1024) { MQ_GEMV(8, 1, false); MQ_GEMV(4, 1, false); MQ_GEMV(2, 1, false); MQ_GEMV(1, 1, false); }
    MQ_GEMV(8, 1, true); MQ_GEMV(4, 1, true); MQ_GEMV(2, 1, true); MQ_GEMV(1, 1, true);
    MQ_GEMV(4, 2, true); MQ_GEMV(2, 2, true); MQ_GEMV(1, 2, true);
    MQ_GEMV(2, 3, true); MQ_GEMV(1, 3, true);
    MQ_GEMV(2, 4, true); MQ_GEMV(1, 4, true);
    MQ_GEMV(1, 6, true); MQ_GEMV(1, 8, true); MQ_GEMV(1, 10, true); MQ_GEMV(1, 12, true);
#undef MQ_GEMV
    return launch_gemv_rows_t<F, 1, 16, true>(x, w, copy_stride, n_copies, scale, y, M, K, reps, stream);
}

}  // namespace mq
