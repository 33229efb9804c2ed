// Prompt-batched prefill: the KV-cache rows of P prompt positions, each layer's
// weights passed over once for all P positions, on the int8 matrix cores.
//
// The reference prefills one decode step per prompt token (a10_decode.py:367-368,
// verify_correctness_a10.py:326-328); the cache rows a step writes are those of
// a10_int8_decode_kernel.cu:143-241. Here the P positions of a chunk go through a
// layer together, as matrix products of P activation rows with each weight matrix.
// The arithmetic is the decode-step kernels' (every stored value is the correctly
// rounded value of the reference's expression, up to fp64 rounding of the sums):
// each activation row becomes a 55-bit fixed-point number over its own
// power-of-two scale (digits.h), the products are exact int32 digit-plane sums
// on the int8 matrix cores recombined in fp64, and attention runs in fp64. So the
// cache rows equal those of P decode steps, apart from fp32 roundings that the
// fp64 summation order can move once in about 2^20 values.
//
// One persistent launch per chunk (a workgroup per compute unit, all resident); per layer
// nine phases over the chunk's P positions, separated by grid barriers:
//   digits      RMSNorm of the layer input (the embedding rows in layer 0), its
//               digit planes                                 one workgroup per position
//   QKV         q|k|v rows on the matrix cores; the epilogue runs QK-norm and RoPE
//               and writes this layer's K/V cache rows and the rotated queries
//               (a 128-row tile is one head, so the norm and the rotation pairs
//               are inside one wave)                        row tiles of 128 (pf_product)
//   attention   causal, fp64 on the matrix cores, per (KV head, 8 positions) its 16
//               queries over cache rows [0, pos0 + p]; a workgroup takes one such
//               item or two of complementary length, its key blocks cut evenly over
//               the four waves
//   digits      of the attention output
//   O           + residual (the layer input)                 row tiles of 64
//   digits      post-attention RMSNorm
//   gate|up     48 channels' gate and up rows per tile; SwiGLU in the epilogue
//   digits      of the SwiGLU output
//   down        + residual, bf16: the next layer's input     row tiles of 32
// The last layer stops after its cache rows. The first generated token comes from
// the decode step of the last prompt token, as in the reference's loop. A phase's work
// items (positions or product tiles) are dealt round-robin over the workgroups.
#include <algorithm>
#include <type_traits>

#include "attention.h"
#include "decode_common.h"
#include "digits.h"

namespace mq {

namespace {

constexpr int kFH = 1024, kFI = 3072, kFD = 128, kFQ = 2048, kFNKV = 8;
constexpr int kFKB = kFI / 64;             // most 64-element K blocks of a product (down: 3072)
constexpr int kTileP = 32;                 // positions per product tile: 4 waves x 4 pairs (or 16: x 2 pairs)
constexpr int kFThreads = 256;
constexpr int kWtBytes = 128 * 1024;       // most weight bytes a product's row tile holds in LDS

// Chunk workspace for Pp positions (a multiple of kTileP). Digit planes are laid out
// [K block of 64][position pair][16 bytes of K][position of the pair][plane][16 bytes]: the
// MFMA A operand of a pair and K block is 1 KB in lane order, so that its load touches each cache
// line once. (As [position][plane][64 bytes] each quarter of a load touched all eight lines: the down
// product, the most load-bound, took 23.0 us at 512 positions and 6.5 at 77, now 17.0 and 4.8.)
struct PfLayout {
    size_t sync, hid, x, q, m, dig, emax, tok, total;
};
constexpr PfLayout pf_layout(size_t Pp) {
    PfLayout o{};
    size_t off = 0;
    o.sync = off; off += 1024;                         // grid-barrier counters, abort flag
    o.hid = off; off += round256(Pp * kFH * 2);        // layer input, bf16
    o.x = off; off += round256(Pp * kFH * 4);          // post-attention residual, fp32
    o.q = off; off += round256(Pp * kFQ * 4);          // rotated queries, fp32
    o.m = off; off += round256(Pp * kFI * 4);          // SwiGLU output, fp32
    o.dig = off; off += round256(Pp * kFKB * 512);     // digit planes of the current product's input
    o.emax = off; off += round256(Pp * 4);             // their exponents, one per position
    o.tok = off; off += round256(Pp * 4);              // the chunk's tokens
    o.total = off;
    return o;
}
constexpr size_t kPfPerPos = pf_layout(1024).total / 1024 + 1;

struct PfArgs {
    const uint16_t* embed;
    const LayerWeights* lw;
    const ScalePointers* sp;
    const uint16_t* cos_t;
    const uint16_t* sin_t;
    uint16_t* kc;
    uint16_t* vc;
    int layer, P, Pp, pos0, S, L;
    float attn_scale;
    uint32_t spin_limit;
    uint8_t* ws;
    uint64_t* trace;                       // optional phase timeline (kPfTracePoints per layer)
};

// Grid-barrier state. Counters are cumulative over a launch (zeroed before it); each XCD has a
// 128-byte cache line of its own.
constexpr int kPfXcd = 8;
constexpr int kPfTracePoints = 18;            // phase k (9 per layer): 2 k phase done, 2 k + 1 barrier passed
struct PfSync {
    struct {
        uint32_t arrived;                  // workgroups of the XCD that reached the current barrier
        uint32_t pad0[7];
        uint32_t released;                 // the last barrier the XCD's leader has passed
        uint32_t pad1[7];
        uint32_t lead;                     // the last barrier the XCD's leader has reached
        uint32_t pad2[7];
        uint32_t abort;                    // xcd[0]'s: set when a barrier wait expired
        uint32_t pad3[7];
    } xcd[kPfXcd];
};
static_assert(sizeof(PfSync) <= 1024, "barrier state");

// LDS of a workgroup, shared by the phases
struct PfShared {
    union {
        double2 am[5][17][kWave];          // attention: the waves' parts of an item (m and denominator, outputs)
        uint4 wt[kWtBytes / 16];           // products: the workgroup's weight rows, as pf_load_weights lays them out
    };
    float sc[128];                         // their row scales
    alignas(16) uint16_t qkg[kFD];                     // QKV: the QK-norm gains of the row tile's head
    alignas(16) uint16_t gain[kFH];                    // RMSNorm gains of the next normed digit phase
    double reds[4];
    uint32_t rede[2][4];                   // the waves' largest exponents, of a workgroup's positions in turn
};

enum PfSrc { SRC_EMBED = 0, SRC_HID = 1, SRC_X = 2, SRC_M = 3, SRC_A = 4 };
enum PfEpi { EPI_QKV = 0, EPI_O = 1, EPI_GU = 2, EPI_DOWN = 3 };

// The kernel runs every phase of every layer in one body. Values that depend only on the
// thread or workgroup index are the same in every layer, and the compiler would otherwise
// compute them once, before the layer loop, and keep them all live through every phase (more
// than the register file holds). Reading the index through an empty volatile asm makes it
// new in each phase, so each phase computes what it needs at its start.
__device__ __forceinline__ int pf_fresh(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

__device__ __forceinline__ int pf_fresh_uniform(int v) {
    asm volatile("" : "+s"(v));
    return v;
}

template <class T>
__device__ __forceinline__ T* pf_buf(const PfArgs& a, size_t off) {
    return reinterpret_cast<T*>(a.ws + off);
}

// x[j] of lane i of each quad becomes x[i] of lane j.
__device__ __forceinline__ void quad_transpose(uint32_t (&x)[4], int lane) {
    auto swap = [&](uint32_t& lo, uint32_t& hi, bool odd, auto ctrl) {
        const uint32_t give = odd ? lo : hi;
        const uint32_t got = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)give, decltype(ctrl)::value, 0xF, 0xF, false);
        if (odd) lo = got;
        else hi = got;
    };
    const std::integral_constant<int, 0xB1> xor1{};        // quad_perm [1,0,3,2]
    const std::integral_constant<int, 0x4E> xor2{};        // quad_perm [2,3,0,1]
    swap(x[0], x[1], lane & 1, xor1);
    swap(x[2], x[3], lane & 1, xor1);
    swap(x[0], x[2], lane & 2, xor2);
    swap(x[1], x[3], lane & 2, xor2);
}

// Digit planes of v (4 consecutive elements k0 .. k0 + 3 of position p, k0 = 4 t for thread t plus
// a multiple of 1024) into the chunk's plane buffer. The quad's four threads hold 16 elements, a
// 16-byte piece of each of the 8 planes, 128 bytes in all: thread j of the quad stores planes 2j
// and 2j + 1.
__device__ __forceinline__ void store_digits4(uint8_t* dig, int Pp, int p, int k0, const float (&v)[4], uint32_t emax,
                                              int lane) {
    int d[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i) digits55(v[i], emax, d[i]);
    uint32_t even[4], odd[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        even[j] = pack4(d[0][2 * j], d[1][2 * j], d[2][2 * j], d[3][2 * j]);
        odd[j] = pack4(d[0][2 * j + 1], d[1][2 * j + 1], d[2][2 * j + 1], d[3][2 * j + 1]);
    }
    quad_transpose(even, lane);
    quad_transpose(odd, lane);
    uint8_t* base = dig + ((size_t)(k0 / 64) * Pp + (p & ~1)) * 512 + 256 * ((k0 % 64) / 16) + 128 * (p & 1) + 32 * (lane & 3);
    reinterpret_cast<uint4*>(base)[0] = make_uint4(even[0], even[1], even[2], even[3]);
    reinterpret_cast<uint4*>(base)[1] = make_uint4(odd[0], odd[1], odd[2], odd[3]);
}

// Largest exponent field over a workgroup of kFThreads threads (uniform result).
__device__ __forceinline__ uint32_t block_max_u32(uint32_t e, uint32_t* red, int wave, int lane, int nwaves) {
    e = wave_max_u32(e);
    if (lane == 0) red[wave] = e;
    __syncthreads();
    uint32_t r = red[0];
    for (int w = 1; w < nwaves; ++w) r = max(r, red[w]);
    return r;
}

// ---- row -> (RMSNorm) -> digit planes ------------------------------------------------
// One work item per position. SRC_EMBED / SRC_HID: the layer input (bf16; in layer 0
// the embedding row of the token, also stored as the layer input), input RMSNorm.
// SRC_X: the post-attention residual, post-attention RMSNorm. SRC_M: the SwiGLU
// output, SRC_A: the attention output (in the query buffer), no norm. The normalized value is fp32(r * rstd * gain) as in the decode
// step (a10_int8_decode_kernel.cu:54-84, :421-457).
// `turn` alternates over a workgroup's positions: an un-normed row has one barrier only, behind
// which a wave may go on to the next position's exponents while another still reads this one's, so
// these have the other half of rede.
template <int K, int SRC>
__device__ void pf_digits(const PfArgs& a, int p, int turn, PfShared& sh) {
    constexpr int G = K / 1024;            // groups of 4 consecutive elements per thread
    static_assert(SRC == SRC_M || SRC == SRC_A || G == 1, "the normed rows are hidden-sized");
    double* const reds = sh.reds;
    uint32_t* const rede = sh.rede[turn];
    const PfLayout L = pf_layout((size_t)a.Pp);
    const int t = pf_fresh(threadIdx.x), lane = t % kWave, wave = t / kWave;
    float v[G][4];
    if constexpr (SRC == SRC_EMBED || SRC == SRC_HID) {
        uint16_t* hid = pf_buf<uint16_t>(a, L.hid) + (size_t)p * kFH;
        const uint16_t* row = hid;
        if constexpr (SRC == SRC_EMBED) row = a.embed + (size_t)pf_buf<int>(a, L.tok)[p] * kFH;
        const uint2 u = *reinterpret_cast<const uint2*>(row + 4 * t);
        if constexpr (SRC == SRC_EMBED) *reinterpret_cast<uint2*>(hid + 4 * t) = u;
        v[0][0] = bf16_bits_to_f32(u.x & 0xffffu);
        v[0][1] = bf16_bits_to_f32(u.x >> 16);
        v[0][2] = bf16_bits_to_f32(u.y & 0xffffu);
        v[0][3] = bf16_bits_to_f32(u.y >> 16);
    } else {
        const float* row = SRC == SRC_X ? pf_buf<float>(a, L.x) + (size_t)p * kFH
                         : SRC == SRC_A ? pf_buf<float>(a, L.q) + (size_t)p * kFQ : pf_buf<float>(a, L.m) + (size_t)p * K;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const float4 f = *reinterpret_cast<const float4*>(row + 1024 * g + 4 * t);
            v[g][0] = f.x; v[g][1] = f.y; v[g][2] = f.z; v[g][3] = f.w;
        }
    }
    float n[G][4];
    if constexpr (SRC != SRC_M && SRC != SRC_A) {
        double ss = 0.0;
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) ss = fma((double)v[g][i], (double)v[g][i], ss);
        ss = wave_sum64(ss);
        if (lane == 0) reds[wave] = ss;
        __syncthreads();
        const double rstd = rms_scale((reds[0] + reds[1]) + (reds[2] + reds[3]), K, kEps);
        // the gains were loaded into LDS a phase ahead (pf_load_gain), but for the launch's first
        const uint16_t* gain = sh.gain;
        if constexpr (SRC == SRC_EMBED) gain = static_cast<const uint16_t*>(a.lw[a.layer].input_layernorm_weight);
        uint2 gu;
        __builtin_memcpy(&gu, gain + 4 * t, 8);      // the first layer's gains at any element offset
        const float gv[4] = {bf16_bits_to_f32(gu.x & 0xffffu), bf16_bits_to_f32(gu.x >> 16),
                             bf16_bits_to_f32(gu.y & 0xffffu), bf16_bits_to_f32(gu.y >> 16)};
#pragma unroll
        for (int i = 0; i < 4; ++i) n[0][i] = (float)((double)v[0][i] * rstd * (double)gv[i]);
    } else {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) n[g][i] = v[g][i];
    }
    uint32_t e = 0;
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i) e = max(e, exp_field(n[g][i]));
    e = block_max_u32(e, rede, wave, lane, kFThreads / kWave);
    uint8_t* dig = pf_buf<uint8_t>(a, L.dig);
#pragma unroll
    for (int g = 0; g < G; ++g) store_digits4(dig, a.Pp, p, 1024 * g + 4 * t, n[g], e, lane);
    if (t == 0) pf_buf<uint32_t>(a, L.emax)[p] = e;
}

// ---- products on the int8 matrix cores -------------------------------------------------
// A workgroup keeps one row tile of the product's weights (ROWS rows, whole K) in LDS and runs
// it against position tiles of 8 NP positions (32 or 16): wave w takes positions [8 NP pt +
// 2 NP w, +2 NP) (NP pairs). Per 64-element K block a wave reads NT B operands (16 weight rows x
// 64 bytes) from LDS and issues NP NT MFMAs on its NP A operands (a pair's 8 + 8 digit planes:
// 1 KB contiguous), which are loaded pf_ring(NP) blocks ahead. Lane n of a block's B operand takes
// tile row pf_row(t, n), so that a lane ends with contiguous rows: 4 of them in each half of a
// head (QKV: the RoPE pairs (i, i + 64) meet in the lane), 4 of O, 3 gate and the same 3 up
// channels, 2 of down. Its values are those of position 2 (2u + h) + l / 32 for pairs (2u, 2u + 1),
// h = bit 4 of l (pair_values). What the epilogue reads is requested before the K loop (residuals,
// RoPE rows) or lies in LDS with the weights (scales, gains). With rows 16 apart in a lane (2-byte
// loads and stores), half of the lanes idle and those reads after the loop, the phases at 512
// positions took QKV 23.6, O 12.7, gate|up 30.7, down 25.9 us; now 16.2, 12.0, 23.6, 24.3.
//
// The weights do not depend on the phases before the product, so their loads are issued while
// the workgroup waits in an earlier grid barrier (pf_load_weights) and cost the product nothing.
// Loaded inside the K loop, three blocks ahead, every load of a wave waited behind them (loads
// return in order; ~4 us from HBM): a tile of 16 K blocks took 20-23 us at any prompt length,
// with 3.4 us of MFMA work. Phases, us at 77 / 512 positions, so loaded -> prefetched into LDS:
// QKV 22.8 / 41.2 -> 8.6 / 23.6, O 24.5 / 25.3 -> 7.6 / 12.7, gate|up 20.4 / 54.6 -> 9.6 / 30.7, down
// 30.7 / 31.4 -> 8.6 / 25.9; the whole prefill 4.40 / 6.77 -> 2.80 / 5.36 ms.
//
// Row tiles, sized for 128 KB of LDS and for every workgroup to hold one: QKV 32 x 128 rows (a
// head each: q heads 0-15, k heads 0-7, v heads 0-7); O 16 x 64 rows; gate|up 64 x (48 gate + 48
// up rows); down 32 x 32 rows.
template <int EPI>
struct GemmShape {
    static constexpr int K = EPI == EPI_O ? kFQ : EPI == EPI_DOWN ? kFI : kFH;
    static constexpr int ROWS = EPI == EPI_QKV ? 128 : EPI == EPI_O ? 64 : EPI == EPI_GU ? 96 : 32;
    static constexpr int NT = ROWS / 16;
    static constexpr int RPL = EPI == EPI_QKV || EPI == EPI_O ? 4 : EPI == EPI_GU ? 3 : 2;   // contiguous rows of a lane
    static constexpr int NRT = EPI == EPI_QKV ? 32 : EPI == EPI_O ? 16 : EPI == EPI_GU ? 64 : 32;
    static_assert(ROWS * K <= kWtBytes, "row tile in LDS");
};
// K blocks whose A operands are in flight (NP = 4 with 8 spills)
constexpr int pf_ring(int np) { return np == 4 ? 4 : 8; }
constexpr int kGuCh = 48;                   // gate|up channels per row tile

// The tile row of block t, lane n.
template <int EPI>
__device__ __forceinline__ int pf_row(int t, int n) {
    constexpr int RPL = GemmShape<EPI>::RPL;
    return 16 * RPL * (t / RPL) + RPL * n + t % RPL;
}

// Bytes of 4 per lane straight into LDS: lane l's word at dst + 4 l.
__device__ __forceinline__ void lds_load4(void* dst, const void* src) {
    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)src,
                                     (void __attribute__((address_space(3)))*)dst, 4, 0, 0);
}

// Row tile rt's weights straight into LDS (no registers held), issued by waves 1-3 (wave 0 is
// polling the grid barrier), and its scales and QK-norm gains, by wave 1; the next grid barrier
// completes them. One instruction takes 8 rows x 128 bytes, whole lines: its 1 KB block in LDS
// holds 16-byte chunk c of row r at slot 8 (r % 8) + (c ^ (r / RPL % 8)), so that the rows that
// eight lanes of a B operand read (RPL apart) lie in different banks.
template <int EPI>
__device__ __forceinline__ void pf_load_weights(const PfArgs& a, int layer, int rt, PfShared& sh) {
    using GS = GemmShape<EPI>;
    constexpr int RG = GS::ROWS / 8, KC = GS::K / 128;
    const int lane = pf_fresh(threadIdx.x) % kWave;
    const int w = __builtin_amdgcn_readfirstlane(pf_fresh(threadIdx.x) / kWave);
    if (w == 0) return;
    // the tile's first row; gate|up: the gate rows', and the up rows' less the gate rows before them
    const LayerWeights* const lw = a.lw + layer;
    const ScalePointers* const sp = a.sp + layer;
    const int8_t* base;
    const int8_t* base_up = nullptr;
    const float* sc;
    const float* sc_up = nullptr;
    if constexpr (EPI == EPI_QKV) {
        const void *q = lw->q_proj_weight, *k = lw->k_proj_weight, *v = lw->v_proj_weight;
        const float *qs = sp->q_scale, *ks = sp->k_scale, *vs = sp->v_scale;
        const int head = rt < 16 ? rt : rt % 8;
        base = static_cast<const int8_t*>(rt < 16 ? q : rt < 24 ? k : v) + (size_t)128 * head * GS::K;
        sc = (rt < 16 ? qs : rt < 24 ? ks : vs) + 128 * head;
        if (w == 1 && rt < 24) {
            const void *qg = lw->q_norm_weight, *kg = lw->k_norm_weight;
            const uint16_t* const gains = static_cast<const uint16_t*>(rt < 16 ? qg : kg) + 2 * lane;
            if ((reinterpret_cast<uintptr_t>(gains) & 2) == 0) {
                lds_load4(sh.qkg, gains);
            } else {                        // a gain vector at an odd element offset
                sh.qkg[2 * lane] = gains[0];
                sh.qkg[2 * lane + 1] = gains[1];
            }
        }
    } else if constexpr (EPI == EPI_GU) {
        base = static_cast<const int8_t*>(lw->gate_proj_weight) + (size_t)kGuCh * rt * GS::K;
        base_up = static_cast<const int8_t*>(lw->up_proj_weight) + ((int64_t)kGuCh * rt - kGuCh) * GS::K;
        sc = sp->gate_scale + kGuCh * rt;
        sc_up = sp->up_scale + (kGuCh * rt - kGuCh);
    } else {
        base = static_cast<const int8_t*>(EPI == EPI_O ? lw->o_proj_weight : lw->down_proj_weight) +
               (size_t)GS::ROWS * rt * GS::K;
        sc = (EPI == EPI_O ? sp->o_scale : sp->down_scale) + GS::ROWS * rt;
    }
    if (w == 1) {
#pragma unroll
        for (int i = 0; i < GS::ROWS; i += kWave) {
            const int r = min(i + lane, GS::ROWS - 1);
            lds_load4(&sh.sc[i], (EPI == EPI_GU && r >= kGuCh ? sc_up : sc) + r);
        }
    }
    const size_t off = (size_t)(lane / 8) * GS::K;
    auto each = [&](auto&& piece) {         // piece(the lane's 16 bytes, their 1 KB block in LDS)
        for (int i = w - 1; i < RG * KC; i += 3) {
            const int g = i / KC, kc = i % KC;
            const int chunk = (lane % 8) ^ (((8 * g + lane / 8) / GS::RPL) % 8);
            const int8_t* const rows = (EPI == EPI_GU && g >= kGuCh / 8 ? base_up : base) + (size_t)8 * g * GS::K;
            piece(rows + off + 128 * kc + 16 * chunk, &sh.wt[(kc * RG + g) * kWave]);
        }
    };
    if (((reinterpret_cast<uintptr_t>(base) | reinterpret_cast<uintptr_t>(base_up)) & 15) == 0) {
        each([&](const int8_t* src, uint4* dst) {
            __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)src,
                                             (void __attribute__((address_space(3)))*)dst, 16, 0, 0);
        });
    } else {                                // weight matrices at any byte offset
        each([&](const int8_t* src, uint4* dst) { __builtin_memcpy(dst + lane, src, 16); });
    }
}

// The RMSNorm gains of the digit phase after next into LDS, by wave 1 inside a grid barrier.
__device__ __forceinline__ void pf_load_gain(const void* gain, PfShared& sh) {
    const int lane = pf_fresh(threadIdx.x) % kWave;
    if (__builtin_amdgcn_readfirstlane(pf_fresh(threadIdx.x) / kWave) != 1) return;
    const uint16_t* const src = static_cast<const uint16_t*>(gain) + 2 * lane;
    if ((reinterpret_cast<uintptr_t>(gain) & 2) == 0) {
#pragma unroll
        for (int i = 0; i < kFH; i += 2 * kWave) lds_load4(&sh.gain[i], src + i);
    } else {                                // a gain vector at an odd element offset
#pragma unroll
        for (int i = 0; i < kFH; i += 2 * kWave) {
            sh.gain[i + 2 * lane] = src[i];
            sh.gain[i + 2 * lane + 1] = src[i + 1];
        }
    }
}

// The exact values of two position pairs' output tiles. Of pair j's tile lane n (< 16) of each
// lane half holds digit sums 0-3 of row n and lane n + 16 sums 4-7 (sum_d S_d 2^(49 - 7d), each
// half exact in fp64); one exchange of 16-lane rows gives lane n pair c0's two halves and lane
// n + 16 pair c1's, so that every lane finishes a value.
__device__ __forceinline__ double pair_values(i32x4_t c0, i32x4_t c1) {
    auto half = [](i32x4_t c) {
        return fma((double)c[0], 2097152.0, fma((double)c[1], 16384.0, fma((double)c[2], 128.0, (double)c[3])));
    };
    const double h0 = half(c0), h1 = half(c1);
    const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)__double2loint(h0), (uint32_t)__double2loint(h1), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)__double2hiint(h0), (uint32_t)__double2hiint(h1), false, false);
    return fma(__hiloint2double((int)hi[0], (int)lo[0]), 268435456.0, __hiloint2double((int)hi[1], (int)lo[1]));
}

// Four bf16 values (8 bytes) at dst.
__device__ __forceinline__ void store_bf16x4(uint16_t* dst, const float (&v)[4]) {
    *reinterpret_cast<uint2*>(dst) =
        make_uint2((uint32_t)f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16),
                   (uint32_t)f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16));
}

template <int EPI, int NP>
__device__ void pf_gemm(const PfArgs& a, int rt, int pt, PfShared& sh) {
    using GS = GemmShape<EPI>;
    constexpr int K = GS::K, NT = GS::NT, NK = K / 64, RG = GS::ROWS / 8, D = pf_ring(NP);
    static_assert(NK % D == 0 && D % 2 == 0, "whole rings");
    const PfLayout L = pf_layout((size_t)a.Pp);
    const int tid = pf_fresh(threadIdx.x), lane = tid % kWave, w = tid / kWave;
    const int p0 = 8 * NP * pt + 2 * NP * w;
    const int l16 = lane % 16, kq = lane / 16;
    // What the epilogue reads of this lane's positions, requested before the K loop
    constexpr int NU = NP / 2;
    const int h = (lane >> 4) & 1;
    int pj[NU];
    uint32_t exv[NU];
    uint2 cs[NU][4];                        // QKV: RoPE rows (cos low, cos high, sin low, sin high half)
    uint2 resh[NU];                         // O: residual (bf16)
    float2 resx[NU];                        // down: residual (fp32)
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        pj[u] = p0 + 2 * (2 * u + h) + (lane >> 5);        // chunk position of this lane's values (< Pp)
        exv[u] = pf_buf<uint32_t>(a, L.emax)[pj[u]];
        if constexpr (EPI == EPI_QKV) {
            const int64_t at = (int64_t)min(a.pos0 + pj[u], a.S - 1) * kFD + 4 * l16;    // clamped into the table
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                __builtin_memcpy(&cs[u][i], a.cos_t + at + 64 * i, 8);       // tables at any element offset
                __builtin_memcpy(&cs[u][2 + i], a.sin_t + at + 64 * i, 8);
            }
        } else if constexpr (EPI == EPI_O) {
            resh[u] = *reinterpret_cast<const uint2*>(pf_buf<uint16_t>(a, L.hid) + (size_t)pj[u] * kFH + 64 * rt + 4 * l16);
        } else if constexpr (EPI == EPI_DOWN) {
            resx[u] = *reinterpret_cast<const float2*>(pf_buf<float>(a, L.x) + (size_t)pj[u] * kFH + 32 * rt + 2 * l16);
        }
    }
    const uint8_t* abase = pf_buf<uint8_t>(a, L.dig) + (size_t)p0 * 512 + 16 * lane;
    const size_t kstride = (size_t)a.Pp * 512;

    i32x4_t A[D][NP];
    auto load = [&](int d) {                // the next K block's A operands into stage d
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const uint4 u = ldg16(abase + 1024 * j);
            A[d][j] = i32x4_t{(int)u.x, (int)u.y, (int)u.z, (int)u.w};
        }
        abase += kstride;
    };
#pragma unroll
    for (int d = 0; d < D; ++d) load(d);
    __builtin_amdgcn_sched_barrier(0);

    // B operand t of K block kb: row pf_row(t, l16), chunk kq + 4 (kb % 2) of 128-byte column kb / 2
    int bat[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int r = pf_row<EPI>(t, l16);
        bat[t] = kWave * (r / 8) + 8 * (r % 8);
    }
    const int ch[2] = {kq ^ (l16 % 8), (kq + 4) ^ (l16 % 8)};
    i32x4_t B[2][NT];
    auto readb = [&](int kb, int odd) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const uint4 u = sh.wt[kWave * RG * (kb / 2) + bat[t] + ch[odd]];
            B[odd][t] = i32x4_t{(int)u.x, (int)u.y, (int)u.z, (int)u.w};
        }
    };
    i32x4_t acc[NP][NT];
#pragma unroll
    for (int j = 0; j < NP; ++j)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[j][t] = i32x4_t{0, 0, 0, 0};
    readb(0, 0);
    for (int kb0 = 0; kb0 < NK; kb0 += D) {
        const bool more = kb0 + D < NK;     // uniform
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int kb = kb0 + d;
            if (d + 1 < D || more) readb(kb + 1, (d + 1) % 2);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < NP; ++j)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[j][t] = mfma_i8(A[d][j], B[d % 2][t], acc[j][t]);
            if (more) load(d);
            // kept in this order: left to itself the scheduler moves later blocks' MFMAs up to
            // the loads and waits for nearly every load in flight before the first of them
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // ---- epilogue ----
    float scv[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) scv[t] = sh.sc[pf_row<EPI>(t, l16)];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int p = pj[u];
        const int e = (int)exv[u] - 181;
        double val[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) val[t] = ldexp(pair_values(acc[2 * u][t], acc[2 * u + 1][t]), e) * (double)scv[t];
        const bool store = p < a.P;
        if constexpr (EPI == EPI_QKV) {
            const int64_t crow = (((int64_t)a.layer * kFNKV + rt % 8) * a.S + (a.pos0 + p)) * kFD;    // K or V cache row
            if (rt < 24) {
                // q or k head: fp32 value, QK RMSNorm over the head's 128 dims (8 in the lane,
                // 16 lanes), RoPE on the pairs (i, i + 64)
                float y[8];
                double ss = 0.0;
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    y[t] = (float)val[t];
                    ss = fma((double)y[t], (double)y[t], ss);
                }
                ss += partner64<1>(ss);
                ss += partner64<2>(ss);
                ss += partner64<4>(ss);
                ss += partner64<8>(ss);
                const double rs = rms_scale(ss, kFD, kEps);
                const uint2 g0 = *reinterpret_cast<const uint2*>(&sh.qkg[4 * l16]);
                const uint2 g1 = *reinterpret_cast<const uint2*>(&sh.qkg[64 + 4 * l16]);
                auto half16 = [](uint2 v, int i) { return bf16_bits_to_f32(((i & 2 ? v.y : v.x) >> (16 * (i & 1))) & 0xffffu); };
                float o0[4], o1[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const double y0 = (double)y[t] * rs * (double)half16(g0, t);
                    const double y1 = (double)y[t + 4] * rs * (double)half16(g1, t);
                    const double cl = half16(cs[u][0], t), ch = half16(cs[u][1], t);
                    const double sl = half16(cs[u][2], t), sh = half16(cs[u][3], t);
                    o0[t] = (float)(y0 * cl - y1 * sl);
                    o1[t] = (float)(y0 * sh + y1 * ch);
                }
                if (store) {
                    if (rt < 16) {
                        float* const qrow = pf_buf<float>(a, L.q) + (size_t)p * kFQ + 128 * rt + 4 * l16;
                        *reinterpret_cast<float4*>(qrow) = make_float4(o0[0], o0[1], o0[2], o0[3]);
                        *reinterpret_cast<float4*>(qrow + 64) = make_float4(o1[0], o1[1], o1[2], o1[3]);
                    } else {
                        store_bf16x4(a.kc + crow + 4 * l16, o0);
                        store_bf16x4(a.kc + crow + 64 + 4 * l16, o1);
                    }
                }
            } else if (store) {
                const float v0[4] = {(float)val[0], (float)val[1], (float)val[2], (float)val[3]};
                const float v1[4] = {(float)val[4], (float)val[5], (float)val[6], (float)val[7]};
                store_bf16x4(a.vc + crow + 4 * l16, v0);
                store_bf16x4(a.vc + crow + 64 + 4 * l16, v1);
            }
        } else if constexpr (EPI == EPI_O) {
            if (store) {
                const float r[4] = {bf16_bits_to_f32(resh[u].x & 0xffffu), bf16_bits_to_f32(resh[u].x >> 16),
                                    bf16_bits_to_f32(resh[u].y & 0xffffu), bf16_bits_to_f32(resh[u].y >> 16)};
                *reinterpret_cast<float4*>(pf_buf<float>(a, L.x) + (size_t)p * kFH + 64 * rt + 4 * l16) =
                    make_float4((float)(val[0] + (double)r[0]), (float)(val[1] + (double)r[1]),
                                (float)(val[2] + (double)r[2]), (float)(val[3] + (double)r[3]));
            }
        } else if constexpr (EPI == EPI_GU) {
            if (store) {
                float* const m = pf_buf<float>(a, L.m) + (size_t)p * kFI + kGuCh * rt + 3 * l16;
#pragma unroll
                for (int t = 0; t < 3; ++t) m[t] = (float)silu_mul(val[t], val[t + 3]);
            }
        } else {
            if (store) {
                const uint32_t lo = f32_to_bf16_bits((float)(val[0] + (double)resx[u].x));
                const uint32_t hi = f32_to_bf16_bits((float)(val[1] + (double)resx[u].y));
                *reinterpret_cast<uint32_t*>(pf_buf<uint16_t>(a, L.hid) + (size_t)p * kFH + 32 * rt + 2 * l16) = lo | (hi << 16);
            }
        }
    }
}

// The product's share of workgroup v: one row tile (the one prefetched, rt = v % NRT) against
// position tiles grp = v / NRT, grp + groups, ... The workgroups are numbered XCD by XCD, so an
// XCD holds few groups: the digit planes of its positions (up to 1.5 MB per 64 positions) stay in
// its L2 while its row tiles pass over them, and what every XCD reads is the weights, during the
// phases before. (With a row tile's groups on one XCD instead, all planes went through every L2:
// the prefill took 2.27 instead of 2.19 ms at 77 positions, 4.58 instead of 4.44 at 512.) A grid smaller than NRT takes its further row tiles' weights inside the phase. Position tiles hold 32 positions or, when that leaves fewer
// rounds' work per workgroup, 16: a 16-position tile takes about 3/5 of a 32-position one's time
// (QKV 8.3 against 13.7 us, gate|up 6.2 against 9.6 us, one tile per workgroup).
template <int EPI>
__device__ __forceinline__ int pf_groups(int G) { return max(G / GemmShape<EPI>::NRT, 1); }

// Workgroup g's place in the order XCD by XCD (workgroups are dealt round-robin over 8 XCDs).
__device__ __forceinline__ int pf_place(int G, int g) { return (g % kPfXcd) * (G / kPfXcd) + g / kPfXcd; }

template <int EPI>
__device__ __forceinline__ bool pf_has_tile(const PfArgs& a, int G, int v) {
    return v / GemmShape<EPI>::NRT < min(pf_groups<EPI>(G), (a.P + 15) / 16);
}

// Issue the loads of workgroup g's row tile of a layer's product.
template <int EPI>
__device__ __forceinline__ void pf_prefetch(const PfArgs& a, int layer, PfShared& sh) {
    const int G = (int)gridDim.x, v = pf_place(G, pf_fresh_uniform((int)blockIdx.x));
    if (pf_has_tile<EPI>(a, G, v)) pf_load_weights<EPI>(a, layer, v % GemmShape<EPI>::NRT, sh);
}

template <int EPI>
__device__ __forceinline__ void pf_product(const PfArgs& a, PfShared& sh) {
    constexpr int NRT = GemmShape<EPI>::NRT;
    const int G = (int)gridDim.x, v = pf_place(G, pf_fresh_uniform((int)blockIdx.x));
    if (!pf_has_tile<EPI>(a, G, v)) return;
    const int groups = pf_groups<EPI>(G), grp = v / NRT;
    const int n32 = (a.P + 31) / 32, n16 = (a.P + 15) / 16;
    const bool small = 3 * ((n16 + groups - 1) / groups) < 5 * ((n32 + groups - 1) / groups);
    for (int rt = v % NRT; rt < NRT; rt += G) {
        if (rt >= G) {                      // not the prefetched tile (uniform)
            __syncthreads();
            pf_load_weights<EPI>(a, a.layer, rt, sh);
            wait_vmem();
            __syncthreads();
        }
        if (small) {
            for (int pt = grp; pt < n16; pt += groups) pf_gemm<EPI, 2>(a, rt, pt, sh);
        } else {
            for (int pt = grp; pt < n32; pt += groups) pf_gemm<EPI, 4>(a, rt, pt, sh);
        }
    }
}

// ---- causal attention on the fp64 matrix cores -------------------------------------------
// Work item (KV head x, tile of 8 positions p0..p0+7): its 16 queries (lane
// column q = lane % 16: position p0 + q % 8, query head 2x + q / 8) attend over the cache
// rows [0, pos0 + p], 16 keys per block, with v_mfma_f64_16x16x4f64 (A: lane l holds
// A[l % 16][l / 16]; B: B[l / 16][l % 16]; D: register i of lane l holds D[4 i + l / 16]
// [l % 16]). Both products are transposed so that each lane works for its own query:
//   scores S^T = K Q^T: A = K (key rows x dim slots), B = Q^T; instruction j's slot g is
//     dim 32 g + j, so lane l reads 32 contiguous dims of key row l % 16 and of its query;
//     register i of lane l then holds key 4 i + g (g = l / 16) of query q;
//   outputs O^T = V^T P^T: A = V^T, B = P^T; instruction j's slot g is key 4 j + g, which
//     is register j of the lane's own scores, and row c of tile t is dim 8 c + t, so lane
//     l reads 8 contiguous dims of V row 4 j + g; register i of tile t then holds dim
//     32 i + 8 g + t of query q.
// Softmax in fp64: e = exp(s - m) with the query's shift m raised only when a block's
// maximum exceeds it by more than 2^8 (then the accumulators are rescaled), so e stays
// below e^256; the lane's partial denominator covers its keys and the four lane groups'
// are added at the end. Each K and V row is read once per item (8 positions share it),
// where the per-position form read it once per position. The outputs (fp32, as the
// reference stores them) replace the item's queries in the query buffer.
typedef double f64x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f64x4_t mfma_f64(double a, double b, f64x4_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// The key blocks [b0, b1) (16 keys each) of item (x, p0) in one wave: the partial softmax
// state of the lane's query over them (shift m, partial denominator lsum, outputs acc, not
// yet divided). An empty range leaves m = -inf, lsum = 0, acc = 0.
__device__ __forceinline__ void pf_attn_blocks(const PfArgs& a, int x, int p0, int b0, int b1, double& m, double& lsum,
                                               f64x4_t (&acc)[8]) {
    const PfLayout L = pf_layout((size_t)a.Pp);
    const int lane = pf_fresh(threadIdx.x) % kWave;
    const int q = lane % 16, g = lane / 16;
    const int pq = p0 + q % 8;                              // chunk position of the lane's query
    const bool qvalid = pq < a.P;
    const int qpos = a.pos0 + pq;                           // its cache position: keys [0, qpos]
    const int klast = a.pos0 + min(p0 + 7, a.P - 1);        // the item's last key
    const double sc = (double)a.attn_scale;
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[t] = f64x4_t{0.0, 0.0, 0.0, 0.0};
    m = -INFINITY;
    lsum = 0.0;
    if (b0 >= b1) return;
    const float* const qrow = pf_buf<float>(a, L.q) + (size_t)min(pq, a.P - 1) * kFQ + 256 * x + 128 * (q / 8);
    double qd[32];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float4 f = qvalid ? reinterpret_cast<const float4*>(qrow + 32 * g)[j] : make_float4(0.f, 0.f, 0.f, 0.f);
        qd[4 * j] = f.x; qd[4 * j + 1] = f.y; qd[4 * j + 2] = f.z; qd[4 * j + 3] = f.w;
    }
    const int64_t head = ((int64_t)a.layer * kFNKV + x) * a.S * kFD;
    const uint16_t* kb = a.kc + head;
    const uint16_t* vb = a.vc + head;
    // K row k0 + q (dims 32 g..), V rows k0 + 4 j + g (dims 8 q..), clamped into the cache;
    // the next block's are in flight while a block is computed
    uint4 kw[4], vw[4];
    auto load = [&](int k0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) kw[j] = ldg16(reinterpret_cast<const uint4*>(kb + (size_t)min(k0 + q, klast) * kFD + 32 * g) + j);
#pragma unroll
        for (int j = 0; j < 4; ++j) vw[j] = ldg16(vb + (size_t)min(k0 + 4 * j + g, klast) * kFD + 8 * q);
    };
    load(16 * b0);
    for (int bk = b0; bk < b1; ++bk) {
        const int k0 = 16 * bk;
        const uint4 kc[4] = {kw[0], kw[1], kw[2], kw[3]};
        const uint4 vc[4] = {vw[0], vw[1], vw[2], vw[3]};
        if (bk + 1 < b1) load(k0 + 16);
        f64x4_t sa = {0.0, 0.0, 0.0, 0.0}, sb = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int j = 0; j < 32; ++j) {
            const uint4 w4 = kc[j / 8];
            const uint32_t w = (j % 8) < 2 ? w4.x : (j % 8) < 4 ? w4.y : (j % 8) < 6 ? w4.z : w4.w;
            const double kv = (j % 2) ? (double)__uint_as_float(w & 0xffff0000u) : (double)bf16_bits_to_f32(w & 0xffffu);
            if (j % 2) sb = mfma_f64(kv, qd[j], sb);
            else sa = mfma_f64(kv, qd[j], sa);
        }
        double e[4], mb = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int key = k0 + 4 * i + g;
            e[i] = (qvalid && key <= qpos) ? (sa[i] + sb[i]) * sc : -INFINITY;
            mb = fmax(mb, e[i]);
        }
        mb = fmax(mb, partner64<16>(mb));
        mb = fmax(mb, partner64<32>(mb));
        // raise the shift when the block's maximum exceeds it by more than 2^8 (always on
        // the first block with a valid key); the same decision in the query's four lanes
        const bool raise = mb > m + 256.0;
        if (__any(raise)) {
            const double alpha = raise ? exp(m - mb) : 1.0;      // 0 while m is -inf
            lsum *= alpha;
#pragma unroll
            for (int t = 0; t < 8; ++t) acc[t] *= alpha;
            m = raise ? mb : m;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            e[i] = e[i] == -INFINITY ? 0.0 : exp(e[i] - m);
            lsum += e[i];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t vv[4] = {vc[j].x, vc[j].y, vc[j].z, vc[j].w};
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const uint32_t w = vv[t / 2];
                const double v = (t % 2) ? (double)__uint_as_float(w & 0xffff0000u) : (double)bf16_bits_to_f32(w & 0xffffu);
                acc[t] = mfma_f64(v, e[j], acc[t]);
            }
        }
    }
}

// Number of 16-key blocks of item (x, p0): keys [0, pos0 + min(p0 + 7, P - 1)].
__device__ __forceinline__ int pf_attn_nblocks(const PfArgs& a, int p0) {
    return (a.pos0 + min(p0 + 7, a.P - 1)) / 16 + 1;
}

// One attention unit on the workgroup's four waves: item A = (KV head x, positions pa ..
// pa + 7) and, if pb >= 0, item B = (x, pb .. pb + 7). The unit's T = nA + nB key blocks (A's,
// then B's) are cut into four contiguous ranges [T w / 4, T (w + 1) / 4), one per wave w, so
// a wave's range may hold the end of A and the start of B. Each part's state goes to LDS: A's
// part of wave w to slot w, B's to slot w + 1 (only one wave can hold both). Then every wave
// merges a quarter of the output dims of each item: all of it in one wave took 2.7 us of a
// short prompt's 11.8. Both workgroup barriers are reached by every wave.
__device__ void pf_attention_unit(const PfArgs& a, int x, int pa, int pb, PfShared& sh) {
    const int w = __builtin_amdgcn_readfirstlane(pf_fresh(threadIdx.x) / kWave);
    const int lane = pf_fresh(threadIdx.x) % kWave;
    const int nA = pf_attn_nblocks(a, pa), nB = pb >= 0 ? pf_attn_nblocks(a, pb) : 0, T = nA + nB;
    auto cut = [&](int i) { return (T * i) / 4; };
    // blocks of wave i's range in item A (k = 0) or B (k = 1): [first, end), counted within the item
    auto first = [&](int k, int i) { return k == 0 ? min(cut(i), nA) : max(cut(i), nA) - nA; };
    auto end = [&](int k, int i) { return k == 0 ? min(cut(i + 1), nA) : max(cut(i + 1), nA) - nA; };
#pragma unroll 1
    for (int k = 0; k < 2; ++k) {
        const int b0 = __builtin_amdgcn_readfirstlane(first(k, w)), b1 = __builtin_amdgcn_readfirstlane(end(k, w));
        if (b0 >= b1) continue;
        double m, lsum;
        f64x4_t acc[8];
        pf_attn_blocks(a, x, k == 0 ? pa : pb, b0, b1, m, lsum, acc);
        double2 (*const slot)[kWave] = sh.am[w + k];
        slot[0][lane] = make_double2(m, lsum);
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
            for (int i = 0; i < 2; ++i) slot[1 + 2 * t + i][lane] = make_double2(acc[t][2 * i], acc[t][2 * i + 1]);
    }
    __syncthreads();
    // wave w: output tiles 2w and 2w + 1 (dims 8 c + 2w, + 1 of the lane's 8-dim runs)
#pragma unroll 1
    for (int k = 0; k < (nB > 0 ? 2 : 1); ++k) {
        double mm = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (first(k, i) < end(k, i)) mm = fmax(mm, sh.am[i + k][0][lane].x);
        double lsum = 0.0, o[2][4] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (first(k, i) >= end(k, i)) continue;
            const double2 ml = sh.am[i + k][0][lane];
            const double f = ml.x == -INFINITY ? 0.0 : exp(ml.x - mm);
            lsum += ml.y * f;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const double2 v = sh.am[i + k][1 + 2 * (2 * w + t) + j][lane];
                    o[t][2 * j] += v.x * f;
                    o[t][2 * j + 1] += v.y * f;
                }
        }
        lsum += partner64<16>(lsum);        // the query's four lanes: all valid or all not
        lsum += partner64<32>(lsum);
        const double r = rcp_nr(lsum);
        const int q = lane % 16, g = lane / 16;
        const int pq = (k == 0 ? pa : pb) + q % 8;
        if (pq < a.P) {
            float* const orow = pf_buf<float>(a, pf_layout((size_t)a.Pp).q) + (size_t)pq * kFQ + 256 * x + 128 * (q / 8);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<float2*>(orow + 32 * i + 8 * g + 2 * w) = make_float2((float)(o[0][i] * r), (float)(o[1][i] * r));
        }
    }
    __syncthreads();                        // the slots are read before the next unit writes them
}

// ---- grid barrier ----------------------------------------------------------------------
// Two levels. A workgroup's results are in its XCD's L2 once it reaches the barrier (each wave
// waits for its own stores first). The last workgroup of an XCD to arrive, counted by an atomic
// that the XCD's L2 performs, is that XCD's leader: its agent-scope release writes the XCD's L2
// back to memory (once per XCD and barrier: one write-back per workgroup, 32 per XCD, cost 26-90
// us per barrier), then it raises its flag, waits for all eight leaders' flags (eight lanes, one
// flag each), acquires at agent scope (its L1 and the L2 drop their stale lines), waits for that,
// and releases its XCD's workgroups through the L2.
// Every other workgroup empties its own L1, which may hold lines of the exchanged buffers as it read
// or wrote them in an earlier phase, with an agent-scope acquire too (no narrower one does it: a
// workgroup-scope acquire is empty where a workgroup runs on one CU). It does so as it arrives, all
// its loads and stores completed, not once it is released: until then the CU reads nothing but
// weights and norm gains, which no phase writes (and not even those in the barrier before attention,
// so that a line they share with a cache row does no harm), so that the L1 holds nothing stale when
// the leader, after the last XCD's write-back, has cleared the L2 and releases it. The acquire
// clears the L2 as well, which costs the phase that is ending less than the one that begins: us of a
// prefill of 2 / 77 / 256 positions with it on arrival 1,986 / 2,292 / 2,775, on release 2,120 /
// 2,389 / 2,877. Barrier number b
// completes when an XCD's arrivals reach b times its workgroups and the flags reach b. A wait
// that expires sets the abort flag, and every later wait of the launch then returns at once,
// so the grid always drains (the host reports MQ_ERR_TIMEOUT, mq_prefill_check). Needs the
// workgroups dealt round-robin over the 8 XCDs (checked by the host).
//
// Waits until every active lane's word has reached the target; runs on a whole wave.
__device__ __forceinline__ bool pf_wait_ge(const uint32_t* p, uint32_t target, PfSync* sy, uint32_t limit) {
    uint32_t n = 0;
    while (__any(__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target)) {
        if (__hip_atomic_load(&sy->xcd[0].abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) return false;
        __builtin_amdgcn_s_sleep(1);
        if (++n >= limit) {
            __hip_atomic_store(&sy->xcd[0].abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
    }
    return true;
}

// `ahead` runs on waves 1-3 while wave 0 waits: it issues the loads of a coming product's weight
// tile into LDS. The last workgroup barrier does not wait for them (lds_barrier: LDS
// operations only); the next grid barrier does.
template <class F>
__device__ __forceinline__ void pf_grid_barrier(PfSync* sy, uint32_t b, uint32_t limit, F&& ahead) {
    wait_vmem();                            // this wave's stores, and its loads into LDS
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(threadIdx.x / kWave) != 0) {
        ahead();
    } else {
        const int lane = threadIdx.x % kWave;
        auto& mine = sy->xcd[hw_xcc_id() % kPfXcd];
        const uint32_t per_xcd = gridDim.x / kPfXcd;
        uint32_t old = 0;
        if (lane == 0) old = __hip_atomic_fetch_add(&mine.arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if ((uint32_t)__builtin_amdgcn_readfirstlane((int)old) == b * per_xcd - 1u) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            if (lane == 0) __hip_atomic_store(&mine.lead, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            pf_wait_ge(&sy->xcd[lane % kPfXcd].lead, b, sy, limit);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            wait_vmem();                    // the lines are gone before the XCD is released
            if (lane == 0) __hip_atomic_store(&mine.released, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        } else {
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            wait_vmem();                    // this CU's L1 is empty
            pf_wait_ge(&mine.released, b, sy, limit);
        }
    }
    lds_barrier();
}

// The whole chunk in one launch: every layer's nine phases, each phase's work items dealt
// over the workgroups: positions round-robin, products as pf_product says, attention items in
// units of even length (pf_attention_unit). A product's weights are requested two barriers
// earlier, in the barrier before the digit phase of its input.
__global__ void __launch_bounds__(kFThreads, 1) pf_chunk_kernel(PfArgs a) {
    __shared__ PfShared sh;
    const PfLayout L0 = pf_layout((size_t)a.Pp);
    PfSync* const sy = pf_buf<PfSync>(a, L0.sync);
    const int G = (int)gridDim.x, g = (int)blockIdx.x;
    uint32_t nb = 0;
    int l = 0;
    auto stamp = [&](int point) {
        if (a.trace != nullptr && threadIdx.x == 0)
            a.trace[((size_t)l * kPfTracePoints + point) * G + g] = __builtin_amdgcn_s_memrealtime();
    };
    auto barrier = [&](int k, auto&& ahead) {
        stamp(2 * k);
        pf_grid_barrier(sy, ++nb, a.spin_limit, ahead);
        stamp(2 * k + 1);
    };
    auto none = [] {};
    pf_prefetch<EPI_QKV>(a, 0, sh);
    for (l = 0; l < a.L; ++l) {
        PfArgs b = a;
        b.layer = l;
        for (int p = pf_fresh_uniform(g), turn = 0; p < a.P; p += G, turn ^= 1) {
            if (l == 0) pf_digits<kFH, SRC_EMBED>(b, p, turn, sh);
            else pf_digits<kFH, SRC_HID>(b, p, turn, sh);
        }
        barrier(0, none);
        pf_product<EPI_QKV>(b, sh);
        if (l == a.L - 1) { stamp(2); break; }                 // the last layer contributes its cache rows only
        barrier(1, none);
        {
            // attention units, one per workgroup: a chunk of at most G items (KV head, tile of 8
            // positions) gives each workgroup one item; a longer one pairs tile j with tile
            // np - 1 - j of the same head, so that every unit holds about as many key blocks.
            // Unit u runs KV head u % 8, on the XCD whose L2 then holds that head's rows.
            const int np = (a.P + 7) / 8, items = kFNKV * np;
            const bool paired = items > G;
            const int units = paired ? kFNKV * ((np + 1) / 2) : items;
            for (int u = pf_fresh_uniform(g); u < units; u += G) {
                const int j = u / kFNKV, jb = np - 1 - j;
                pf_attention_unit(b, u % kFNKV, 8 * j, paired && jb > j ? 8 * jb : -1, sh);
            }
        }
        barrier(2, [&] { pf_prefetch<EPI_O>(a, l, sh); });
        for (int p = pf_fresh_uniform(g), turn = 0; p < a.P; p += G, turn ^= 1) pf_digits<kFQ, SRC_A>(b, p, turn, sh);
        barrier(3, [&] { pf_load_gain(a.lw[l].post_attn_layernorm_weight, sh); });
        pf_product<EPI_O>(b, sh);
        barrier(4, [&] { pf_prefetch<EPI_GU>(a, l, sh); });
        for (int p = pf_fresh_uniform(g), turn = 0; p < a.P; p += G, turn ^= 1) pf_digits<kFH, SRC_X>(b, p, turn, sh);
        barrier(5, none);
        pf_product<EPI_GU>(b, sh);
        barrier(6, [&] { pf_prefetch<EPI_DOWN>(a, l, sh); });
        for (int p = pf_fresh_uniform(g), turn = 0; p < a.P; p += G, turn ^= 1) pf_digits<kFI, SRC_M>(b, p, turn, sh);
        barrier(7, [&] { if (l + 1 < a.L) pf_load_gain(a.lw[l + 1].input_layernorm_weight, sh); });
        pf_product<EPI_DOWN>(b, sh);
        barrier(8, [&] { pf_prefetch<EPI_QKV>(a, l + 1, sh); });
    }
}

__global__ void pf_sync_reset_kernel(PfSync* sy) {
    sy->xcd[0].abort = 0u;
    for (int x = 0; x < kPfXcd; ++x) {
        sy->xcd[x].arrived = 0u;
        sy->xcd[x].released = 0u;
        sy->xcd[x].lead = 0u;
    }
}

__global__ void pf_sync_status_kernel(const PfSync* sy, uint32_t* out) { *out = sy->xcd[0].abort; }

}  // namespace

size_t prefill_workspace_bytes(int max_tokens) {
    if (max_tokens < 1) return 0;
    const size_t Pp = (size_t)(max_tokens + kTileP - 1) / kTileP * kTileP;
    return pf_layout(Pp).total;
}

// Positions one chunk holds in `bytes` of workspace (a multiple of kTileP), 0 if none.
int prefill_capacity(size_t bytes) {
    size_t Pp = bytes / kPfPerPos / kTileP * kTileP;
    while (Pp >= (size_t)kTileP && pf_layout(Pp).total > bytes) Pp -= kTileP;
    return (int)std::min(Pp, (size_t)1 << 20);
}

// The chunk kernel's grid: one workgroup per compute unit (its barriers need every workgroup
// resident; checked with the occupancy calculator).
static int prefill_grid(int* grid) {
    static thread_local int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return set_error(MQ_ERR_HIP, "hipGetDevice failed");
    if (cached[dev] == 0) {
        int ncu = 0, per_cu = 0;
        if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(&pf_chunk_kernel),
                                                         kFThreads, 0) != hipSuccess)
            return set_error(MQ_ERR_HIP, "occupancy query failed");
        if (ncu < kPfXcd || ncu % kPfXcd != 0 || per_cu < 1 || !xcd_placement_ok())
            return set_error(MQ_ERR_UNSUPPORTED, "the prefill kernel needs its workgroups dealt round-robin over "
                             "8 XCDs (%d compute units)", ncu);
        cached[dev] = ncu;
    }
    *grid = cached[dev];
    return MQ_OK;
}

int launch_prefill(const mq_decode_args& d, const int* tokens, int n_tokens, void* ws, size_t ws_bytes,
                   hipStream_t stream) {
    const int cap = prefill_capacity(ws_bytes);
    if (cap < kTileP) return set_error(MQ_ERR_INVALID_ARGUMENT, "prefill workspace of %zu bytes holds no chunk", ws_bytes);
    int grid = 0;
    int st = prefill_grid(&grid);
    if (st != MQ_OK) return st;
    PfArgs a{};
    a.embed = static_cast<const uint16_t*>(d.embed_weight);
    a.lw = d.layer_weights;
    a.sp = d.scales;
    a.cos_t = static_cast<const uint16_t*>(d.cos_table);
    a.sin_t = static_cast<const uint16_t*>(d.sin_table);
    a.kc = static_cast<uint16_t*>(d.k_cache);
    a.vc = static_cast<uint16_t*>(d.v_cache);
    a.S = d.max_seq_len;
    a.L = d.num_layers;
    a.attn_scale = d.attn_scale;
    a.spin_limit = d.spin_limit ? d.spin_limit : (1u << 21);
    a.ws = static_cast<uint8_t*>(ws);
    a.trace = static_cast<uint64_t*>(d.trace);
    a.Pp = cap;
    const PfLayout L = pf_layout((size_t)cap);
    PfSync* sy = reinterpret_cast<PfSync*>(a.ws + L.sync);
    for (int c0 = 0; c0 < n_tokens; c0 += cap) {
        a.P = std::min(cap, n_tokens - c0);
        a.pos0 = d.position + c0;
        const hipError_t e = hipMemcpyAsync(a.ws + L.tok, tokens + c0, (size_t)a.P * sizeof(int),
                                            hipMemcpyHostToDevice, stream);
        if (e != hipSuccess) return set_error(MQ_ERR_HIP, "hipMemcpyAsync(prefill tokens): %s", hipGetErrorString(e));
        // a fill kernel, not a memset, so that the launch sequence can be captured in a graph
        pf_sync_reset_kernel<<<1, 1, 0, stream>>>(sy);
        void* args[] = {&a};
        const hipError_t le = launch_resident(reinterpret_cast<const void*>(&pf_chunk_kernel), dim3(grid),
                                              dim3(kFThreads), args, stream);
        if (le != hipSuccess) return set_error(MQ_ERR_HIP, "launch(prefill): %s", hipGetErrorString(le));
        st = check_launch("prefill");
        if (st != MQ_OK) return st;
    }
    return MQ_OK;
}

int prefill_check(void* ws, size_t ws_bytes, hipStream_t stream) {
    const int cap = prefill_capacity(ws_bytes);
    if (cap < kTileP) return set_error(MQ_ERR_INVALID_ARGUMENT, "prefill workspace of %zu bytes holds no chunk", ws_bytes);
    uint32_t* flag = nullptr;
    if (hipHostMalloc(reinterpret_cast<void**>(&flag), sizeof(uint32_t), hipHostMallocDefault) != hipSuccess)
        return set_error(MQ_ERR_HIP, "hipHostMalloc failed");
    *flag = 0u;
    const PfLayout L = pf_layout((size_t)cap);
    pf_sync_status_kernel<<<1, 1, 0, stream>>>(reinterpret_cast<const PfSync*>(static_cast<uint8_t*>(ws) + L.sync), flag);
    int st = check_launch("prefill check");
    if (st == MQ_OK && hipStreamSynchronize(stream) != hipSuccess) st = set_error(MQ_ERR_HIP, "hipStreamSynchronize failed");
    const uint32_t v = *flag;
    (void)hipHostFree(flag);
    if (st != MQ_OK) return st;
    return v ? set_error(MQ_ERR_TIMEOUT, "a grid barrier of the prefill expired (were all compute units free?)") : MQ_OK;
}

}  // namespace mq
