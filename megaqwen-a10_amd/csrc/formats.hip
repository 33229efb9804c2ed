// Other weight formats on gfx950: FP8 E4M3 per-row and INT4 per-group weight-only
// matvecs, and their quantizers from bf16. The reference has INT8 (bench_int8.py:19-24)
// and BF16 weights only; these follow the INT8 quantizer's pattern (symmetric scale
// from the absolute maximum, IEEE division, round half to even) with:
//   FP8  (OCP E4M3FN, decoded by v_cvt_pk_f32_fp8): per row s = fp32(amax) / 448,
//        q = nearest code of fp32(w) / s (ties to the even code, |x| >= 448 -> +-448)
//   INT4 per group of 128 elements of a row: s = bf16(amax / 7), q = clamp(rint(w / s), -8, 7),
//        two's complement nibbles, low nibble = even element
// Matvecs y[j] = sum_k dequant(w)[j, k] x[k], fp32 x and y.
//   FP8: the row kernel of gemv_rows.h, as the INT8 matvec: 8 v_cvt_pk_f32_fp8 per 16 weights,
//        fp32 accumulation, the row scale applied after the row sum.
//   INT4: on the int8 matrix cores, as the decode step's products: x as a 55-bit fixed-point
//        vector in eight digit planes, the biased nibbles as the int8 operand, exact integer
//        sums per group of 128, recombined and scaled in fp64 (int4_gemv_kernel).
#include "common.h"
#include "digits.h"
#include "gemv_rows.h"
#include "internal.h"
#include "quant_rows.h"

#include <algorithm>

namespace mq {

namespace {

constexpr int kFmtThreads = 256;
constexpr int kFmtWaves = kFmtThreads / kWave;
constexpr int kInt4Group = 128;

// ---- quantizers: rows that quant_rows.h does not take (odd lengths, unaligned views, few FP8 rows) ----
__device__ __forceinline__ float block_max_abs(float v, float* red) {
    v = wave_max(v);
    const int wave = threadIdx.x / kWave;
    if ((threadIdx.x % kWave) == 0) red[wave] = v;
    __syncthreads();
    float m = red[0];
#pragma unroll
    for (int i = 1; i < kFmtWaves; ++i) m = fmaxf(m, red[i]);
    return m;
}

__global__ void __launch_bounds__(kFmtThreads)
quantize_fp8_rows_kernel(const uint16_t* __restrict__ w, int64_t K, uint8_t* __restrict__ q, float* __restrict__ scale) {
    const int64_t row = blockIdx.x;
    const uint16_t* wr = w + row * K;
    uint8_t* qr = q + row * K;
    __shared__ float red[kFmtWaves];
    float amax = 0.0f;
    for (int64_t k = threadIdx.x; k < K; k += kFmtThreads) amax = fmaxf(amax, fabsf(bf16_bits_to_f32(wr[k])));
    const float m = block_max_abs(amax, red);
    const float s = fmaxf(__fdiv_rn(m, 448.0f), 1e-12f);
    if (threadIdx.x == 0) scale[row] = s;
    for (int64_t k = threadIdx.x; k < K; k += kFmtThreads)
        qr[k] = (uint8_t)fp8_e4m3_encode(__fdiv_rn(bf16_bits_to_f32(wr[k]), s));
}

// One workgroup per row; thread t quantizes groups t, t + 256, ... of the row.
__global__ void __launch_bounds__(kFmtThreads)
quantize_int4_groups_kernel(const uint16_t* __restrict__ w, int64_t K, uint8_t* __restrict__ q,
                            float* __restrict__ scale) {
    const int64_t row = blockIdx.x;
    const int64_t ng = K / kInt4Group;
    for (int64_t gi = threadIdx.x; gi < ng; gi += kFmtThreads) {
        const uint16_t* wg = w + row * K + gi * kInt4Group;
        float amax = 0.0f;
        for (int k = 0; k < kInt4Group; ++k) amax = fmaxf(amax, fabsf(bf16_bits_to_f32(wg[k])));
        const float s = fmaxf(round_bf16(__fdiv_rn(amax, 7.0f)), 1e-12f);
        scale[row * ng + gi] = s;
        uint8_t* qg = q + row * (K / 2) + gi * (kInt4Group / 2);
        for (int k = 0; k < kInt4Group; k += 2) {
            const float r0 = fminf(fmaxf(__builtin_rintf(__fdiv_rn(bf16_bits_to_f32(wg[k]), s)), -8.0f), 7.0f);
            const float r1 = fminf(fmaxf(__builtin_rintf(__fdiv_rn(bf16_bits_to_f32(wg[k + 1]), s)), -8.0f), 7.0f);
            qg[k / 2] = (uint8_t)(((uint32_t)(int)r0 & 15u) | (((uint32_t)(int)r1 & 15u) << 4));
        }
    }
}

// ---- matvecs -----------------------------------------------------------------------------
// ---- INT4 matvec on the int8 matrix cores ----------------------------------------------------
// y[j] = sum_g s[j, g] sum_{k in g} q[j, k] x[k], with the decode step's exact products: x
// becomes X_k = trunc(x_k 2^(181 - emax)) (emax the largest biased exponent of x; |X_k| <
// 2^55) held as eight 7-bit digit planes in LDS. Each nibble is taken biased, b = n XOR 8 =
// q + 8 in [0, 15], as the int8 operand, so that unpacking is two masks a word. Per group of
// 128 elements two v_mfma_i32_16x16x64_i8 give the exact digit sums sum_k b_k d_p(X_k) of 16
// rows; they are recombined in fp64 (one rounding), corrected by -8 S_g with S_g = sum_{k in
// g} X_k (exact int64, once per workgroup), scaled by s[j, g] and summed over the groups in
// fp64; y = fp32(2^(emax - 181) sum). Besides fp64 roundings the error is x's truncation
// to 55 bits of its largest element (x finite).
//
// Operands. For group g, lane (n, kq) (n = lane % 16, kq = lane / 16) of a wave item (16 rows
// from row0) needs the 16 bytes of row row0 + n holding elements 128 g + 32 kq + [0, 32), as
// words w0..w3 of 8 nibbles. K step h (0, 1) of the group takes {lo(w_2h), hi(w_2h),
// lo(w_2h+1), hi(w_2h+1)} as the B operand (lo: the even nibbles masked into bytes, hi: the
// odd ones), so byte j of the lane's 16 holds element 128 g + 32 kq + 16 h + e(j), e = 0 2 4
// 6 1 3 5 7 8 10 12 14 9 11 13 15. Digit plane p holds its digit of that element at byte
// 128 g + 64 h + 16 kq + j (int4_plane_byte), so the A operand of lane l is 16 contiguous
// bytes of plane (l % 16) & 7. Rows 8-15 of the A operand repeat planes 0-7: their sums land
// in lanes 32-63, which are not read. Planes are K + 16 bytes apart, so that the eight
// planes' reads fall on different LDS banks.
//
// Loads. The rows' bytes come in pairs of groups (128 bytes of a row): load A takes rows 0-7
// of the item, load B rows 8-15, lane l chunk c = kq + 4 ((l >> 3) & 1) (16 bytes) of the pair,
// so that every load instruction reads whole 128-byte lines; one row_ror:8 exchange then
// hands lane (n, kq) chunk kq of row n for the pair's first group and chunk kq + 4 for its
// second. The scales of a row are contiguous and only lanes 0-15 (where the row sums end)
// use them: 16-byte loads of four groups' scales when K / 128 is a multiple of 4. (16 rows of
// 64 bytes per load, and one 4-byte scale load per group, measured 0.50-0.56 of the HBM
// peak at the Qwen3-0.6B shapes; this form 0.69-0.81.)
//
// Work. A workgroup takes tiles of 16 rows, each cut along K over S of its waves (whole pairs
// of groups). The waves' fp64 partial sums of a tile meet in LDS and are added in wave order. A
// wave requests its first tile's weights before the workgroup forms the digit planes. Where there
// are tiles enough for eight waves a CU, a wave takes whole tiles instead, one after the other
// (no prefetch: its registers would cost one wave in five, [1024, 2048] in a stream of matvecs
// 0.179 -> 0.190 us). Planes are formed from four or eight consecutive elements per thread. Without the
// cut, and with the planes formed first, byte by byte, from one element per load, calls took (us,
// matrices read in turn) [1024, 3072] 16.0, [2048, 6144] 29.9, [12288, 2048] 12.2, [6144, 1024] 7.0,
// [151936, 1024] 27.4; now 6.3, 8.4, 9.8, 5.6 and 19.1.
// A row's planes take 8 K bytes of LDS, so past 7.8 K elements a CU holds one or two workgroups: these
// have up to 16 waves between them, and tiles are cut until a CU has that many. With four waves each,
// [16384, 16384] 85 us, [28672, 8192] 52; now 35 and 42 (in a stream of matvecs 51 and 29, now 29 and 23).
constexpr int kW4Unroll = 4;                      // group pairs whose loads are issued together
constexpr int kW4MaxWaves = 16;

// Byte of element k (k % 8 == 0) in a digit plane; elements k .. k + 7 follow it in the order
// 0 2 4 6 1 3 5 7.
__device__ __forceinline__ int int4_plane_byte8(int k) {
    const int r = k & 127;
    return (k & ~127) + 64 * ((r >> 4) & 1) + 16 * (r >> 5) + (r & 8);
}

// x's digit planes and group sums into LDS, E (4 or 8) consecutive elements per thread, a thread's
// first ones in registers between the two passes. Returns emax; a barrier must follow.
template <int E>
__device__ __forceinline__ uint32_t int4_planes(const float* __restrict__ x, int K, uint8_t* planes, int PS, double* sg,
                                                uint32_t* red, int lane, int wave) {
    const int threads = blockDim.x;
    float xv[E];
    auto load = [&](int k) {
#pragma unroll
        for (int i = 0; i < E; i += 4) {
            const float4 f = *reinterpret_cast<const float4*>(x + k + i);
            xv[i] = f.x; xv[i + 1] = f.y; xv[i + 2] = f.z; xv[i + 3] = f.w;
        }
    };
    uint32_t em = 0;
    for (int k = E * (int)threadIdx.x; k < K; k += E * threads) {
        load(k);
#pragma unroll
        for (int i = 0; i < E; ++i) em = max(em, exp_field(xv[i]));
    }
    const bool one = K <= E * threads;            // xv still holds them
    em = wave_max_u32(em);
    if (lane == 0) red[wave] = em;
    __syncthreads();
    for (int i = 0; i < threads / kWave; ++i) em = max(em, red[i]);
    for (int k = E * (int)threadIdx.x; k < K; k += E * threads) {
        if (!one) load(k);
        uint64_t X[E];
        int64_t t = 0;
#pragma unroll
        for (int i = 0; i < E; ++i) {
            X[i] = (uint64_t)fixed55(xv[i], em);
            t += (int64_t)X[i];
        }
        uint8_t* const at = planes + int4_plane_byte8(k & ~7) + ((k & 4) >> 1);
#pragma unroll
        for (int p = 0; p < 8; ++p) {             // digit p as digits55 has it, a plane at a time (registers)
            uint32_t d[E];
#pragma unroll
            for (int i = 0; i < E; ++i) {
                d[i] = (uint32_t)(X[i] >> (49 - 7 * p)) & 127u;
                if (p == 0) d[i] = (d[i] ^ 64u) - 64u;              // the top digit is signed
            }
            if constexpr (E == 8) {
                *reinterpret_cast<uint2*>(at + p * PS) =
                    make_uint2(pack4(d[0], d[2], d[4], d[6]), pack4(d[1], d[3], d[5], d[7]));
            } else {
                *reinterpret_cast<uint16_t*>(at + p * PS) = (uint16_t)((d[0] & 0xffu) | (d[2] << 8));
                *reinterpret_cast<uint16_t*>(at + p * PS + 4) = (uint16_t)((d[1] & 0xffu) | (d[3] << 8));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // S_g: 128 / E consecutive threads hold a group
#pragma unroll
        for (int o = 1; o < kInt4Group / E; o <<= 1) t += __shfl_xor(t, o, kInt4Group / E);
        if ((k & (kInt4Group - 1)) == 0) sg[k / kInt4Group] = (double)t;
    }
    return em;
}

// A tile's rows as a lane reads them: pA + 128 q and pB + 128 q its chunks of pair q, srow its row's
// scales (rows past M repeat the last one; they are never stored).
struct Int4Rows {
    const uint8_t *pA, *pB;
    const float* srow;
    int64_t yrow;                                 // its row of y
    bool valid;
};
__device__ __forceinline__ Int4Rows int4_rows(const uint8_t* w, int64_t copy_stride, int n_copies, const float* scale, int M,
                                              int K, int nt, int it, int lane) {
    const int rep = (int)((uint32_t)it / (uint32_t)nt), tile = it - rep * nt;     // it < 2^31
    const int copy = (int)((uint32_t)rep % (uint32_t)n_copies);
    const int c = (lane >> 4) + 4 * ((lane >> 3) & 1);
    const uint8_t* const wc = w + (int64_t)copy * copy_stride + 16 * c;
    const int rA = min(16 * tile + (lane & 7), M - 1), rB = min(16 * tile + 8 + (lane & 7), M - 1);
    const int row = 16 * tile + (lane & 15);
    return {wc + (int64_t)rA * (K / 2), wc + (int64_t)rB * (K / 2), scale + (int64_t)min(row, M - 1) * (K / kInt4Group),
            (int64_t)copy * M + row, row < M};
}

// The chunks of pairs q0 .. q0 + U - 1 that lie below pair p1 (kCut) and below group ng.
template <bool kCut>
__device__ __forceinline__ void int4_load(const Int4Rows& r, int q0, int p1, int ng, int lane, uint4 (&va)[kW4Unroll],
                                          uint4 (&vb)[kW4Unroll]) {
#pragma unroll
    for (int u = 0; u < kW4Unroll; ++u) {
        if ((!kCut || q0 + u < p1) && 2 * (q0 + u) + ((lane >> 3) & 1) < ng) {      // the group this lane's chunk is in
            va[u] = ldg16_stream(r.pA + 128 * (q0 + u));
            vb[u] = ldg16_stream(r.pB + 128 * (q0 + u));
        }
    }
}

// Adds the scaled sums of these pairs' groups to acc (row n in lane n < 16).
template <bool kCut>
__device__ __forceinline__ void int4_pairs(const uint4 (&va)[kW4Unroll], const uint4 (&vb)[kW4Unroll], const float* srow,
                                           int q0, int p1, int ng, bool vec_scales, const uint8_t* arow, const double* sg,
                                           int lane, double& acc) {
    constexpr int U = kW4Unroll;
    const bool low = (lane & 8) == 0;
    float sc[2 * U];
    if (vec_scales && (!kCut || (q0 & 1) == 0) && 2 * (q0 + U) <= ng) {             // 16-byte aligned
#pragma unroll
        for (int u = 0; u < 2 * U; u += 4) {
            float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
            if (lane < 16) f = *reinterpret_cast<const float4*>(srow + 2 * q0 + u);
            sc[u] = f.x; sc[u + 1] = f.y; sc[u + 2] = f.z; sc[u + 3] = f.w;
        }
    } else {
#pragma unroll
        for (int u = 0; u < 2 * U; ++u)
            sc[u] = ((!kCut || q0 + u / 2 < p1) && 2 * q0 + u < ng) ? srow[2 * q0 + u] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < 2 * U; ++u) {
        const int g = 2 * q0 + u;
        if ((!kCut || q0 + u / 2 < p1) && g < ng) {
            // first group of the pair: low lanes keep their A chunk, high lanes take B from
            // lane - 8; second group: low lanes take A from lane + 8, high lanes keep B
            const uint4& mine = (u & 1) ? vb[u / 2] : va[u / 2];
            const uint4& other = (u & 1) ? va[u / 2] : vb[u / 2];
            const bool keep = (u & 1) ? !low : low;
            auto pick = [&](uint32_t m, uint32_t o) -> uint32_t {
                const uint32_t r = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)o, 0x128, 0xF, 0xF, false);
                return keep ? m : r;                               // 0x128: row_ror:8
            };
            const uint32_t q0w = pick(mine.x, other.x) ^ 0x88888888u, q1w = pick(mine.y, other.y) ^ 0x88888888u;
            const uint32_t q2w = pick(mine.z, other.z) ^ 0x88888888u, q3w = pick(mine.w, other.w) ^ 0x88888888u;
            const i32x4_t b0 = {(int)(q0w & 0x0F0F0F0Fu), (int)((q0w >> 4) & 0x0F0F0F0Fu),
                                (int)(q1w & 0x0F0F0F0Fu), (int)((q1w >> 4) & 0x0F0F0F0Fu)};
            const i32x4_t b1 = {(int)(q2w & 0x0F0F0F0Fu), (int)((q2w >> 4) & 0x0F0F0F0Fu),
                                (int)(q3w & 0x0F0F0F0Fu), (int)((q3w >> 4) & 0x0F0F0F0Fu)};
            const uint4 a0 = *reinterpret_cast<const uint4*>(arow + kInt4Group * g);
            const uint4 a1 = *reinterpret_cast<const uint4*>(arow + kInt4Group * g + 64);
            i32x4_t cc = mfma_i8(i32x4_t{(int)a0.x, (int)a0.y, (int)a0.z, (int)a0.w}, b0, i32x4_t{0, 0, 0, 0});
            cc = mfma_i8(i32x4_t{(int)a1.x, (int)a1.y, (int)a1.z, (int)a1.w}, b1, cc);
            // lane n: digits 0-3 of row n, lane n + 16: digits 4-7 (each sum < 2^18, exact)
            const double half = ((double)cc[0] * 2097152.0 + (double)cc[1] * 16384.0) +
                                ((double)cc[2] * 128.0 + (double)cc[3]);
            const double v = fma(half, 268435456.0, partner64<16>(half)) - 8.0 * sg[g];
            acc = fma(v, (double)sc[u], acc);
        }
    }
}

// kCut: tiles cut over S waves, the first tile's weights requested first; otherwise whole tiles in
// workgroups of four waves.
template <bool kCut>
__global__ void __launch_bounds__(kCut ? kW4MaxWaves * kWave : kFmtThreads)
int4_gemv_kernel(const float* __restrict__ x, const uint8_t* __restrict__ w, int64_t copy_stride, int n_copies,
                 const float* __restrict__ scale, float* __restrict__ y, int M, int K, int reps, int S, bool vec_scales) {
    extern __shared__ __align__(16) uint8_t w4lds[];
    __shared__ uint32_t red[kW4MaxWaves];
    __shared__ double part[2][kW4MaxWaves][16];
    constexpr int U = kW4Unroll;
    const int PS = K + 16;                        // digit plane stride in bytes
    uint8_t* const planes = w4lds;
    double* const sg = reinterpret_cast<double*>(w4lds + 8 * PS);   // S_g of each group
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int ng = K / kInt4Group, np = (ng + 1) / 2;               // groups, pairs of groups
    const int nt = (M + 15) / 16;
    const int items = reps * nt;                  // < 2^31, checked by the host
    auto rows = [&](int it) { return int4_rows(w, copy_stride, n_copies, scale, M, K, nt, it, lane); };

    // kCut: the workgroup's tiles at once, the wave's tile among them and its pairs of that
    const int tiles = kCut ? (int)blockDim.x / kWave / S : 0, slot = kCut ? wave / S : 0, seg = kCut ? wave % S : 0;
    const int p0 = kCut ? np * seg / S : 0, p1 = kCut ? np * (seg + 1) / S : np;
    int base = blockIdx.x * tiles;                // first tile of the workgroup's round
    Int4Rows r;
    uint4 fa[U], fb[U];
    if (kCut && base + slot < items) {
        r = rows(base + slot);
        int4_load<kCut>(r, p0, p1, ng, lane, fa, fb);
    }
    // eight elements per thread leave most threads of a short row without any
    const uint32_t em = K <= 1024 ? int4_planes<4>(x, K, planes, PS, sg, red, lane, wave)
                                  : int4_planes<8>(x, K, planes, PS, sg, red, lane, wave);
    __syncthreads();

    const uint8_t* const arow = planes + (lane & 7) * PS + 16 * (lane >> 4);
    const double unit = ldexp(1.0, (int)em - 181);
    if constexpr (!kCut) {
        const int total_waves = gridDim.x * kFmtWaves;
        for (int it = blockIdx.x * kFmtWaves + wave; it < items; it += total_waves) {
            r = rows(it);
            double acc = 0.0;
            for (int q0 = 0; q0 < np; q0 += U) {
                uint4 va[U], vb[U];
                int4_load<kCut>(r, q0, np, ng, lane, va, vb);
                int4_pairs<kCut>(va, vb, r.srow, q0, np, ng, vec_scales, arow, sg, lane, acc);
            }
            if (lane < 16 && r.valid) y[r.yrow] = (float)(acc * unit);
        }
    } else {
        int round = 0;
        for (bool ahead = true; base < items; base += gridDim.x * tiles, round ^= 1, ahead = false) {
            const int it = base + slot;
            double acc = 0.0;
            if (it < items) {
                if (!ahead) r = rows(it);
                for (int q0 = p0; q0 < p1; q0 += U) {
                    if (!ahead || q0 != p0) int4_load<kCut>(r, q0, p1, ng, lane, fa, fb);
                    int4_pairs<kCut>(fa, fb, r.srow, q0, p1, ng, vec_scales, arow, sg, lane, acc);
                }
            }
            // the waves' partial sums of a tile, added in order by its first wave; two buffers, so
            // that one barrier a round is enough
            if (lane < 16) part[round][wave][lane] = acc;
            __syncthreads();
            if (seg == 0 && it < items && lane < 16) {
                for (int i = 1; i < S; ++i) acc += part[round][wave + i][lane];
                if (r.valid) y[r.yrow] = (float)(acc * unit);
            }
        }
    }
}

int launch_int4_t(const float* x, const uint8_t* w, int64_t copy_stride, int n_copies, const float* scale, float* y,
                  int M, int K, int reps, hipStream_t stream) {
    const int64_t items = (int64_t)reps * ((M + 15) / 16);
    const int np = (K / kInt4Group + 1) / 2;
    auto lds_bytes = [](size_t k) { return 8 * (k + 16) + sizeof(double) * (k / kInt4Group); };
    const size_t lds = lds_bytes((size_t)K);
    const int64_t cus = device_cu_count();
    const int fit = (int)(163840 / (lds + 4352));        // workgroups whose planes (and 4 KB) fit a CU's LDS
    const bool wide = fit <= 2;                          // these share 16 waves between them
    // waves per tile: enough for eight waves a CU (16 where the LDS holds few workgroups), each with a
    // pair of groups at least, then no more than the waves that this leaves the same most pairs
    int S = (int)std::min<int64_t>(((wide ? 16 : 8) * cus + items - 1) / items, std::min(np, kW4MaxWaves));
    const int per = (np + S - 1) / S;
    S = (np + per - 1) / per;
    const int tiles = std::max(1, (wide ? 16 / fit : 4) / S);         // tiles a workgroup works on at once
    const int threads = S * tiles * kWave;
    const bool cut = S > 1 || wide;
    // workgroups at once: as many as fit, with cut tiles at most 16 waves a CU, otherwise five of the
    // uncut kernel's by its registers; each with the same number of tiles, in whole workgroups per CU
    // (in a stream of matvecs [4096, 1024] 0.35 us, with eight a CU, of which three wait, 0.38; [1024, 1024]
    // 0.100, with 1171 workgroups instead of 1280 0.109)
    const int64_t most = wide ? fit * cus : cut ? std::max<int64_t>(1, 16 * cus / (S * tiles)) : std::min(fit, 5) * cus;
    const int64_t want = (items + tiles - 1) / tiles;
    const int64_t rounds = (want + most - 1) / most;
    const int64_t even = (want + rounds - 1) / rounds;
    const int grid = (int)(rounds > 1 ? (even + cus - 1) / cus * cus : even);
    const auto kernel = cut ? int4_gemv_kernel<true> : int4_gemv_kernel<false>;
    if (lds > 57344) {                             // with the kernel's static 4 KB past the default limit
        static bool raised[2][64] = {};            // per device: the limit is the current device's
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
        if (!raised[cut][dev]) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes(16384));
            if (e != hipSuccess) return set_error(MQ_ERR_HIP, "int4_gemv: %zu bytes of LDS: %s", lds, hipGetErrorString(e));
            raised[cut][dev] = true;
        }
    }
    const bool vec_scales = ((uintptr_t)scale % 16) == 0 && (K / kInt4Group) % 4 == 0;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), lds, stream,
                       x, w, copy_stride, n_copies, scale, y, M, K, reps, S, vec_scales);
    return check_launch("int4_gemv");
}

}  // namespace

// Fewer rows than four per CU leave a wave per row too few waves to hide the encoding of its codes
// (some 20 instructions each), and a workgroup per row is faster: [64, 8192] 9.8 us against 13.0,
// [512, 4096] 6.8 / 8.1, [512, 1024] 3.9 / 4.1; [1024, 8192] 15.2 / 15.2, [1024, 2048] 5.9 / 5.5. (INT8's
// and INT4's codes are cheaper: [64, 8192] 9.2 / 6.9 and 14.6 / 9.6.)
int launch_quantize_fp8(const void* w_bf16, int M, int K, uint8_t* q, float* scale, hipStream_t stream) {
    if (M >= 4 * device_cu_count() && quant_rows_fit(w_bf16, K, q, 8)) {
        launch_quant_rows<Q_FP8>(w_bf16, M, K, q, scale, device_cu_count(), stream);
        return check_launch("quantize_fp8");
    }
    hipLaunchKernelGGL(quantize_fp8_rows_kernel, dim3(M), dim3(kFmtThreads), 0, stream,
                       static_cast<const uint16_t*>(w_bf16), (int64_t)K, q, scale);
    return check_launch("quantize_fp8_rows_kernel");
}

int launch_quantize_int4(const void* w_bf16, int M, int K, uint8_t* q, float* scale, hipStream_t stream) {
    if (quant_rows_fit(w_bf16, K, q, 4)) {
        launch_quant_rows<Q_INT4>(w_bf16, M, K, q, scale, device_cu_count(), stream);
        return check_launch("quantize_int4");
    }
    hipLaunchKernelGGL(quantize_int4_groups_kernel, dim3(M), dim3(kFmtThreads), 0, stream,
                       static_cast<const uint16_t*>(w_bf16), (int64_t)K, q, scale);
    return check_launch("quantize_int4_groups_kernel");
}

int launch_fp8_gemv(const float* x, const uint8_t* w, int64_t copy_stride, int n_copies, const float* scale, float* y,
                    int M, int K, int reps, hipStream_t stream) {
    return launch_gemv_rows<Fp8W>(x, w, copy_stride, n_copies, scale, y, M, K, reps, stream);
}

int launch_int4_gemv(const float* x, const uint8_t* w, int64_t copy_stride, int n_copies, const float* scale, float* y,
                     int M, int K, int reps, hipStream_t stream) {
    return launch_int4_t(x, w, copy_stride, n_copies, scale, y, M, K, reps, stream);
}

}  // namespace mq
