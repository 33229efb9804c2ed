// Weight-only matvec of one-byte weights with per-row scales, y[j] = scale[j] * sum_k x[k] *
// w[j,k] (INT8: gemv.hip, FP8: formats.hip), fp32 activations and sums.
//
// Layout: one 64-lane wave owns R consecutive rows at a time; each lane reads 16 contiguous
// weights of a row per 1 KB chunk (a coalesced 1 KB row segment per wave instruction) and holds
// the activations of its own 16 columns of every chunk in registers for all its rows. The R row
// sums are finished with a transpose reduction (R values -> 1 per lane group).
//
// Bound by memory: HBM for large matrices, and for a few MB one memory round trip, so a wave
// requests its first rows before anything else, the activations (L2 after the first wave) right
// behind them, and each further item's rows while it computes the one before. No LDS and no
// workgroup barrier. (The activations staged through LDS by the workgroup, element by element,
// before the first weight load: kernel times at [2048, 6144] 10.5 us against 7.2 now, [12288, 2048]
// 8.9 / 7.3, [1024, 3072] 4.5 / 3.7, [1024, 2048] 3.9 / 3.3.) The weights are streamed past the
// last-level cache, where a model's other matrices would displace them anyway: [151936, 1024] 30.9 ->
// 28.0 us a call.
// R is the largest for the row length (R rows x chunks of 16 bytes per lane in flight) that
// still gives every CU two workgroups of items, so that small shapes spread over every CU.
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
constexpr int kGemvPerCu = 4;     // LM head [151936, 1024]: 2 workgroups a CU 32.4 us, 4 28.0, 8 28.6

// F::dot(w, x, acc): 16 weights against x[0..3], the activations of elements 4 i .. 4 i + 3.
template <class F, int R, int CHMAX>
__global__ void __launch_bounds__(kGemvThreads)
gemv_rows_kernel(const float* __restrict__ x, const uint8_t* __restrict__ w, int64_t copy_stride, int n_copies,
                 const float* __restrict__ scale, float* __restrict__ y, int M, int K, int reps) {
    const int lane = threadIdx.x % kWave;
    const int total_waves = gridDim.x * kGemvWaves;
    const int nbatch = (M + R - 1) / R;
    const int64_t items = (int64_t)reps * nbatch;
    int64_t it = blockIdx.x * kGemvWaves + threadIdx.x / kWave;
    uint4 next[R][CHMAX];
    auto load = [&](int64_t i) {
        const int rep = (int)(i / nbatch);
        const int row0 = (int)(i - (int64_t)rep * nbatch) * R;
        const uint8_t* const wc = w + (int64_t)(rep % n_copies) * copy_stride;
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < CHMAX; ++c) {
                next[r][c] = make_uint4(0, 0, 0, 0);
                const int col = c * 1024 + lane * 16;
                if (row0 + r < M && col < K) next[r][c] = ldg16_stream(wc + (int64_t)(row0 + r) * K + col);
            }
    };
    if (it < items) load(it);
    float4 xv[CHMAX][4];
#pragma unroll
    for (int c = 0; c < CHMAX; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int col = c * 1024 + lane * 16;
            xv[c][i] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (col < K) xv[c][i] = reinterpret_cast<const float4*>(x + col)[i];
        }
    for (; it < items; it += total_waves) {
        uint4 wv[R][CHMAX];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < CHMAX; ++c) wv[r][c] = next[r][c];
        if (it + total_waves < items) load(it + total_waves);
        float acc[R];
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = 0.0f;
#pragma unroll
        for (int c = 0; c < CHMAX; ++c)
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r] = F::dot(wv[r][c], xv[c], acc[r]);
        const float s = transpose_reduce<R>(acc, lane);
        constexpr int span = kWave / R;
        const int rep = (int)(it / nbatch);
        const int row = (int)(it - (int64_t)rep * nbatch) * R + lane / span;
        if ((lane % span) == 0 && row < M) y[(int64_t)(rep % n_copies) * M + row] = s * scale[row];
    }
}

template <class F, int R, int CHMAX>
int launch_gemv_rows_t(const float* x, const uint8_t* w, int64_t copy_stride, int n_copies, const float* scale, float* y,
                       int M, int K, int reps, hipStream_t stream) {
    const int64_t items = (int64_t)reps * ((M + R - 1) / R);
    // at most kGemvPerCu workgroups a CU, and no more waves than give each the same number of items,
    // in whole workgroups per CU: [151936, 1024] with 950 workgroups on 256 CUs took 28.0 us a call (INT8)
    // and 27.4 (FP8), with 1024 27.2 and 26.6 (three alternating runs, spread 0.15 at most)
    const int64_t most = (int64_t)kGemvPerCu * device_cu_count() * kGemvWaves;
    const int64_t per = (items + most - 1) / most;
    const int64_t waves = (items + per - 1) / per;
    const int64_t cus = device_cu_count(), even = (waves + kGemvWaves - 1) / kGemvWaves;
    const int grid = (int)(per > 1 ? (even + cus - 1) / cus * cus : even);
    hipLaunchKernelGGL((gemv_rows_kernel<F, R, CHMAX>), dim3(grid), dim3(kGemvThreads), 0, stream,
                       x, w, copy_stride, n_copies, scale, y, M, K, reps);
    return check_launch("gemv_rows_kernel");
}

template <class F>
int launch_gemv_rows(const float* x, const uint8_t* w, int64_t copy_stride, int n_copies, const float* scale, float* y,
                     int M, int K, int reps, hipStream_t stream) {
    const int CH = (K + 1023) / 1024;
    int R = CH <= 1 ? 8 : CH == 2 ? 4 : CH <= 4 ? 2 : 1;
    const int64_t min_waves = (int64_t)2 * kGemvWaves * device_cu_count();
    while (R > 1 && (int64_t)reps * ((M + R - 1) / R) < min_waves) R /= 2;
#define MQ_GEMV(RR, CC)                                                                                            \
    if (CH <= CC && R == RR) return launch_gemv_rows_t<F, RR, CC>(x, w, copy_stride, n_copies, scale, y, M, K, reps, stream)
    MQ_GEMV(8, 1); MQ_GEMV(4, 1); MQ_GEMV(2, 1); MQ_GEMV(1, 1);
    MQ_GEMV(4, 2); MQ_GEMV(2, 2); MQ_GEMV(1, 2);
    MQ_GEMV(2, 3); MQ_GEMV(1, 3);
    MQ_GEMV(2, 4); MQ_GEMV(1, 4);
    MQ_GEMV(1, 6); MQ_GEMV(1, 8);
#undef MQ_GEMV
    return launch_gemv_rows_t<F, 1, 16>(x, w, copy_stride, n_copies, scale, y, M, K, reps, stream);
}

}  // namespace mq
