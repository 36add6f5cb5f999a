// AWQ W4A16 for a decode batch up to a short prompt: packed weights streamed into LDS, unpacked once per block for up to 128 tokens.
//
// Between one 16-token MFMA tile and a large GEMM the op is bound by neither HBM nor the matrix cores but by what is done per weight: unpacking
// (1 to 2 vector instructions a weight) and the LDS traffic of unpacked weights.  Here
//   * a block owns a column tile of 32 packed words (256 channels, one 128-byte line per row of the weight matrix) and up to 128 tokens.  Its
//     wavefronts come in K slices of four: each slice walks its own share of K in stages of 64 rows through a ring of LDS stages that are
//     filled by direct loads (global_load_lds: packed weights, activations, scales and zero points alike), several stages ahead;
//   * a wavefront of a slice owns one byte of every word, i.e. two of its eight channels: it reads the eight words of a lane's MFMA operand
//     (8 consecutive k of one word column), v_perm_b32 picks its byte from two k-adjacent words, and two channels x 8 k come out as the
//     operands of v_mfma_f32_32x32x16_f16.  Nothing is unpacked twice in a block, and unpacked weights never go through LDS;
//   * a lane keeps its word column in the accumulators too (tokens are the row operand), so a group's scale is one value per lane.
// FOLD: (q - z) enters the matrix core as an exact small integer and the group's sum is scaled in fp32, the arithmetic of the few-token
// kernel (awq_decode.hip); otherwise fp16((q - z) s), the reference's rounding, as in the tile kernel (awq_tile.hip).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "awq_plans.h"
#include "llmq_common.h"

namespace llmq {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

constexpr int kStageK = 64;                   // rows of the weight matrix per LDS stage
constexpr int kTileWords = 32;                // packed words per column tile: one 128-byte line a row
constexpr int kTileCh = 8 * kTileWords;
constexpr int kOutStride = 2 * kTileCh + 16;  // bytes between the token rows of the finished tile in LDS
constexpr int kWBytes = kStageK * kTileWords * 4, kSBytes = 2 * kTileWords * 16, kZBytes = 2 * kTileWords * 4;

struct StreamArgs {
    const uint16_t* x;       // [M, K], row stride ldx elements
    const uint32_t* qw;      // [K, N / 8]
    const uint16_t* scales;  // [K / G, N]
    const uint32_t* qz;      // [K / G, N / 8]
    const uint16_t* bias;    // [N] fp16 or null
    uint16_t* out;           // [M, N]
    float* partials;         // splits > 1: one block of accumulators per (split, token slab, column tile)
    int64_t ldx;
    int M, N, K;
    int halves_per_group;    // G / 32
    uint32_t group_mul;      // ceil(2^32 / halves_per_group)
    int units_per_block;     // K range of a block, in units of the kernel
    int tiles_n, splits, slabs;
};

template <int MT_, int KS_, int NS_, bool FOLD_, bool BF_, int V_>
struct StreamCfg {
    static constexpr int MT = MT_;          // 32-token tiles per block
    static constexpr int KS = KS_;          // K slices: sets of four wavefronts with LDS stages of their own
    static constexpr int NS = NS_;          // LDS stages per slice
    static constexpr bool FOLD = FOLD_;     // group sums scaled in fp32; groups of whole units
    static constexpr bool BF = BF_;         // x and out are bf16 (rounded to fp16 on the way in, the fp16 result widened)
    static constexpr int V = V_;            // packed words per direct load: 4 (rows of whole 16-byte pieces) or 1
    static constexpr int UNIT = FOLD ? 2 : 1;                       // stages per unit of K
    static constexpr int WL = (V == 4 ? 8 : 32) / 4;                // weight loads per wavefront and stage
    static constexpr int LPT = WL + MT;                             // ... and of activations; scales or zero points are one more
    static constexpr int X_AT = kWBytes, S_AT = X_AT + MT * 4096, Z_AT = S_AT + kSBytes, STAGE_BYTES = Z_AT + kZBytes;
    static constexpr int Q = 2 * MT * 4;                            // accumulator quads of a lane
    static constexpr int NT = 256 * KS;
    static constexpr int LDS_BYTES = KS * NS * STAGE_BYTES;
    static_assert(LDS_BYTES <= 160 * 1024 && (NS - 1) * (LPT + 1) < 64, "LDS of a CU; vmcnt is a 6-bit counter");
    static_assert((KS - 1) * Q * 4096 <= LDS_BYTES && 32 * MT * kOutStride <= LDS_BYTES && Q % KS == 0, "the epilogue reuses the stages");
};

__device__ __forceinline__ u4 to_f16x8(u4 v) {
    u4 r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t w = v[i];
        r[i] = Lo<LLMQ_F16>::pack2(Lo<LLMQ_BF16>::lo_f32(w), Lo<LLMQ_BF16>::hi_f32(w));
    }
    return r;
}
// the finished value of one output: fp16(sum), then fp16(that + bias), then widened for a bf16 model
template <bool BF>
__device__ __forceinline__ uint16_t finish_value(float v, bool has_bias, float bias) {
    uint16_t h = Lo<LLMQ_F16>::from_f32(v);
    if (has_bias) h = Lo<LLMQ_F16>::from_f32(Lo<LLMQ_F16>::to_f32(h) + bias);
    return BF ? Lo<LLMQ_BF16>::from_f32(Lo<LLMQ_F16>::to_f32(h)) : h;
}
__device__ __forceinline__ int channel_of(int byte, int p) { return 4 * (byte & 1) + (byte >> 1) + 2 * p; }  // nibble 2 byte + p of a word

template <class C>
__global__ __launch_bounds__(C::NT, 2) void awq_stream_kernel(StreamArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr int MT = C::MT, KS = C::KS, NS = C::NS;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave_b = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int slice = wave_b >> 2, wv = wave_b & 3;  // wv: the byte of a word that this wavefront unpacks
    const int l32 = lane & 31, khalf = lane >> 5;
    const int Nw = a.N >> 3;

    // Flat block ids go round-robin over the 8 XCDs; each XCD gets a run of consecutive (K split, column tile, token slab) triples, as many as
    // the others: the slabs of a column tile share its weights through one L2.  (With all slabs of a tile on one XCD, whatever that did to the
    // balance, 245 blocks of 819 x 8832 x 18176 put 35 on some XCDs of 32 CUs: 459 us instead of 247.)
    const int xcd = blockIdx.x & 7, q8 = gridDim.x >> 3, r8 = gridDim.x & 7;
    const int pid = xcd * q8 + min(xcd, r8) + (blockIdx.x >> 3);
    const int slab = pid % a.slabs, work = pid / a.slabs, tile = work % a.tiles_n, split = work / a.tiles_n;
    const int m0 = slab * 32 * MT, rows = min(32 * MT, a.M - m0);

    // ---- this slice's stages
    const int units = a.K / (kStageK * C::UNIT);
    const int b_begin = split * a.units_per_block, b_cnt = min(units, b_begin + a.units_per_block) - b_begin;
    const int per = (b_cnt + KS - 1) / KS;
    const int u_begin = b_begin + min(slice * per, b_cnt), u_end = b_begin + min((slice + 1) * per, b_cnt);
    const int s0 = u_begin * C::UNIT, ns = (u_end - u_begin) * C::UNIT;  // first stage, number of stages (0: an empty slice)
    const int n_block = per * C::UNIT;                                   // barriers are block-wide

    // ---- direct loads.  A wavefront's 64 pieces land back to back in LDS; which global piece lands where is free per lane.
    // Weights: LDS row slot 16 c + 2 r + h holds row 16 c + r + 8 h of the stage, so that the two half-waves of an operand read (rows r and
    // r + 8) touch 256 consecutive bytes.
    const uint32_t lds_base = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)smem) + (uint32_t)(slice * NS * C::STAGE_BYTES);
    uint32_t w_off;
    if constexpr (C::V == 4) {
        const int l8 = lane >> 3;
        w_off = 4u * (uint32_t)(((l8 >> 1) + 8 * (l8 & 1)) * Nw + min(tile * kTileWords + 4 * (lane & 7), Nw - 4));
    } else {
        w_off = 4u * (uint32_t)(8 * khalf * Nw + min(tile * kTileWords + l32, Nw - 1));
    }
    uint32_t x_off[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int row = (wv * MT + i) * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
        x_off[i] = 2u * (uint32_t)(min(row, rows - 1) * (int)a.ldx + 8 * piece);
    }
    const int cw = tile * kTileWords + l32, cwc = min(cw, Nw - 1);
    const uint16_t* xb = a.x + (int64_t)m0 * a.ldx;
    auto issue = [&](int s, int slot) __attribute__((always_inline)) {  // s: stage of this slice
        const int sa = s0 + s;
        const uint32_t dst = lds_base + (uint32_t)(slot * C::STAGE_BYTES);
        const uint32_t* wb = a.qw + (int64_t)sa * kStageK * Nw;
#pragma unroll
        for (int i = 0; i < C::WL; i++) {
            const int g = wv * C::WL + i;  // 1 KB (V = 4: 8 row slots) or 256 bytes (2 row slots) of the stage
            const uint32_t* src = wb + (int64_t)(C::V == 4 ? (g >> 1) * 16 + (g & 1) * 4 : (g >> 3) * 16 + (g & 7)) * Nw;
            const uint32_t m0v = dst + (uint32_t)g * (C::V == 4 ? 1024u : 256u);
            if constexpr (C::V == 4)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0v), "v"(w_off), "s"(src) : "memory", "m0");
            else
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(m0v), "v"(w_off), "s"(src) : "memory", "m0");
        }
        const uint16_t* xs = xb + sa * kStageK;
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const uint32_t m0v = dst + (uint32_t)(C::X_AT + (wv * MT + i) * 1024);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0v), "v"(x_off[i]), "s"(xs) : "memory", "m0");
        }
        if (C::FOLD && (s & 1)) return;  // (a unit's group comes with its first stage)
        // scales and zero points of the two 32-row halves of the stage; two wavefronts fetch either, so that all issue the same number
        const uint32_t half = 2u * (uint32_t)sa + (uint32_t)khalf;
        const uint32_t g = a.halves_per_group == 1 ? half : __umulhi(half, a.group_mul);
        const uint32_t m0v = dst + (uint32_t)((wv & 1) ? C::Z_AT : C::S_AT);
        if (wv & 1) {
            const uint32_t off = 4u * (g * (uint32_t)Nw + (uint32_t)cwc);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(m0v), "v"(off), "s"(a.qz) : "memory", "m0");
        } else {
            const uint32_t off = 16u * (g * (uint32_t)Nw + (uint32_t)cwc);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0v), "v"(off), "s"(a.scales) : "memory", "m0");
        }
    };
    // this wavefront's loads of stage t have landed when only those of `younger` later stages of its are in flight; odd_c: t is odd
    auto wait_stage = [&](int younger, auto odd_c) __attribute__((always_inline)) {
        constexpr bool odd = decltype(odd_c)::value;
        auto loads = [](int n) constexpr { return n * C::LPT + (C::FOLD ? (odd ? n + 1 : n) / 2 : n); };  // of stages t + 1 .. t + n
        constexpr int kA = loads(NS - 1), kB = loads(NS - 2), kC = loads(1);
        if (younger >= NS - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kA) : "memory");
        else if (younger >= NS - 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kB) : "memory");
        else if (NS > 3 && younger == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kC) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    static_assert(NS <= 4, "wait_stage tells 0, 1, NS - 2 and NS - 1 younger stages apart");
    uint8_t* ring = smem + slice * NS * C::STAGE_BYTES;
    // bf16 activations become fp16 in place, each wavefront the pieces that it loaded: read, and a sub-step later written back
    u4 piece[C::BF ? MT : 1];
    auto convert_read = [&](int slot) __attribute__((always_inline)) {
        const u4* p = reinterpret_cast<const u4*>(ring + slot * C::STAGE_BYTES + C::X_AT + wv * MT * 1024) + lane;
#pragma unroll
        for (int i = 0; i < MT; i++) piece[C::BF ? i : 0] = p[i * kWave];
    };
    auto convert_write = [&](int slot) __attribute__((always_inline)) {
        u4* p = reinterpret_cast<u4*>(ring + slot * C::STAGE_BYTES + C::X_AT + wv * MT * 1024) + lane;
#pragma unroll
        for (int i = 0; i < MT; i++) p[i * kWave] = to_f16x8(piece[C::BF ? i : 0]);
    };
    auto lds_barrier = []() __attribute__((always_inline)) {  // orders LDS traffic only: the loads stay in flight across it
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    v16f acc[2][MT], y[2][C::FOLD ? MT : 1];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                acc[p][i][r] = 0.f;
                if (C::FOLD) y[p][C::FOLD ? i : 0][r] = 0.f;
            }

    const uint32_t sel = (uint32_t)wv | 0x0c00u | ((uint32_t)(4 + wv) << 16) | 0x0c000000u;
    uint32_t magic = 0x64006400u;
    asm volatile("" : "+v"(magic));  // opaque: (u & mask) | magic stays one v_and_or_b32
    const h2 k16 = {(_Float16)0.0625f, (_Float16)0.0625f};

    // ---- software pipeline over sub-steps of 16 k: packed words are read two sub-steps ahead, unpacked one ahead, activations read one ahead,
    // all of it dealt out between the MFMAs.  (Left to itself the compiler read each pair of words right before its use, one LDS latency per pair.)
    struct Raw { uint32_t w[8], z; uint2 s; };  // z, s: with the first sub-step of a stage half (FOLD: of a unit)
    struct Op { uint32_t lo[4], hi[4]; };
    Raw raw[2];
    Op op[2];
    h8 xa[2][MT];
    h2 czl, czh, sl, sh;
    float f0 = 0.f, f1 = 0.f;  // FOLD: the scales of the unit in the accumulators
    uint2 s_next = {0u, 0u};   // ... and of the one being unpacked
    // sub-steps that start a new group's zero points and scales
    auto new_group = [](auto ks_c, auto odd_c) { return std::integral_constant<bool, decltype(ks_c)::value % 2 == 0 && (!C::FOLD || (decltype(ks_c)::value == 0 && !decltype(odd_c)::value))>{}; };
    auto read_words = [&](const uint8_t* st, int ks, int pr, Raw& r) __attribute__((always_inline)) {  // k pair pr of sub-step ks
        const uint32_t* W = reinterpret_cast<const uint32_t*>(st) + lane;
        r.w[2 * pr] = W[(16 * ks + 4 * pr) * kTileWords];
        r.w[2 * pr + 1] = W[(16 * ks + 4 * pr + 2) * kTileWords];
    };
    auto read_group = [&](const uint8_t* st, int ks, Raw& r) __attribute__((always_inline)) {
        r.z = *reinterpret_cast<const uint32_t*>(st + C::Z_AT + 4 * ((ks >> 1) * kTileWords + l32));
        r.s = *reinterpret_cast<const uint2*>(st + C::S_AT + 16 * ((ks >> 1) * kTileWords + l32) + 8 * (wv & 1));
    };
    auto read_x = [&](const uint8_t* st, int ks, int i, h8* f) __attribute__((always_inline)) {
        const int row = 32 * i + l32;
        f[i] = __builtin_bit_cast(h8, reinterpret_cast<const u4*>(st + C::X_AT)[row * 8 + ((2 * ks + khalf) ^ ((row >> 1) & 7))]);
    };
    auto start_group = [&](const Raw& r) __attribute__((always_inline)) {
        const uint32_t z = r.z >> (8 * wv);
        czl = __builtin_bit_cast(h2, (0xE400u | (z & 0xFu)) * 0x00010001u);   // -(1024 + z)
        czh = __builtin_bit_cast(h2, (0xD400u | (z & 0xF0u)) * 0x00010001u);  // -(64 + z)
        if constexpr (C::FOLD) {
            s_next = r.s;
        } else {
            const uint32_t pick = (wv >> 1) ? 0x03020302u : 0x01000100u;
            sl = __builtin_bit_cast(h2, __builtin_amdgcn_perm(r.s.x, r.s.x, pick));
            sh = __builtin_bit_cast(h2, __builtin_amdgcn_perm(r.s.y, r.s.y, pick));
        }
    };
    auto unpack = [&](const Raw& r, int pr, Op& o) __attribute__((always_inline)) {
        const uint32_t u = __builtin_amdgcn_perm(r.w[2 * pr + 1], r.w[2 * pr], sel);  // byte 0 <- k 2 pr, byte 2 <- k 2 pr + 1
        h2 l = __builtin_bit_cast(h2, (u & 0x000F000Fu) | magic) + czl;                                 // (1024 + q) - (1024 + z)
        h2 h = __builtin_elementwise_fma(__builtin_bit_cast(h2, (u & 0x00F000F0u) | magic), k16, czh);  // (1024 + 16 q) / 16 - (64 + z)
        if constexpr (!C::FOLD) l = l * sl, h = h * sh;
        o.lo[pr] = __builtin_bit_cast(uint32_t, l);
        o.hi[pr] = __builtin_bit_cast(uint32_t, h);
        asm volatile("" : "+v"(o.lo[pr]), "+v"(o.hi[pr]));  // here, between the MFMAs: the compiler sank a sub-step's unpacking behind the barrier
    };
    auto fold_tile = [&](int p, int i) __attribute__((always_inline)) {  // FOLD: a finished group sum times the group's scale
        const float f = p ? f1 : f0;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            float t = fmaf(f, acc[p][i][r], y[p][C::FOLD ? i : 0][r]);
            asm volatile("" : "+v"(t));  // here and not later: moved, the sums of two groups are live at once (54 registers more, spills)
            y[p][C::FOLD ? i : 0][r] = t;
        }
    };
    auto next_scales = [&]() __attribute__((always_inline)) {
        f0 = Lo<LLMQ_F16>::to_f32((uint16_t)((wv >> 1) ? s_next.x >> 16 : s_next.x & 0xffffu));
        f1 = Lo<LLMQ_F16>::to_f32((uint16_t)((wv >> 1) ? s_next.y >> 16 : s_next.y & 0xffffu));
    };
    // Sub-step `ks` of the stage `st`: its MFMAs; between them the words of the sub-step after next (stage rw_st) and the activations of the next
    // one (stage rx_st) are read and the next one's words unpacked.  START (FOLD): the accumulators hold the last unit's sums, which are folded
    // tile by tile as they restart.  odd: stage of a unit.
    auto sub_step = [&](auto ks_c, auto odd_c, const uint8_t* rw_st, const uint8_t* rx_st) __attribute__((always_inline)) {
        constexpr int ks = decltype(ks_c)::value, SLOTS = 2 * MT;
        constexpr bool ODD = decltype(odd_c)::value, START = C::FOLD && ks == 0 && !ODD;
        constexpr int ks1 = (ks + 1) & 3, ks2 = (ks + 2) & 3;
        constexpr bool odd1 = ks + 1 < 4 ? ODD : (C::FOLD && !ODD), odd2 = ks + 2 < 4 ? ODD : (C::FOLD && !ODD);
        const Op& o = op[ks & 1];
        Op& on = op[(ks + 1) & 1];
        const Raw& rn = raw[(ks + 1) & 1];
        Raw& r2 = raw[ks & 1];
        const h8* f = xa[ks & 1];
        h8* fn = xa[(ks + 1) & 1];
        const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        const h8 bl = __builtin_bit_cast(h8, v4i{(int)o.lo[0], (int)o.lo[1], (int)o.lo[2], (int)o.lo[3]});
        const h8 bh = __builtin_bit_cast(h8, v4i{(int)o.hi[0], (int)o.hi[1], (int)o.hi[2], (int)o.hi[3]});
#pragma unroll
        for (int m = 0; m < SLOTS; m++) {
            const int p = m / MT, i = m % MT;
            if constexpr (START) fold_tile(p, i);
            acc[p][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[i], p ? bh : bl, START ? zero : acc[p][i], 0, 0, 0);
            if (m < MT && ks != 2) read_x(rx_st, ks1, m, fn);  // (those of sub-step 3 are read before the barrier)
            if (m == 0 && decltype(new_group(std::integral_constant<int, ks1>{}, std::integral_constant<bool, odd1>{}))::value) start_group(rn);
#pragma unroll
            for (int pr = 0; pr < 4; pr++)
                if (pr * SLOTS / 4 == m) unpack(rn, pr, on), read_words(rw_st, ks2, pr, r2);
            if (m == SLOTS - 1 && decltype(new_group(std::integral_constant<int, ks2>{}, std::integral_constant<bool, odd2>{}))::value) read_group(rw_st, ks2, r2);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (START) next_scales();
    };

    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    // Stage kt is computed while kt + 1 .. kt + NS - 1 are in flight; its slot takes stage kt + NS as soon as its last words are read, in the
    // middle of the stage, where the barrier also publishes stage kt + 1.
#pragma unroll
    for (int t = 0; t < NS; t++)
        if (t < ns) issue(t, t);
    wait_stage(min(ns, NS) - 1, std::false_type{});
    if (C::BF && ns > 0) convert_read(0), convert_write(0);
    lds_barrier();
#pragma unroll
    for (int pr = 0; pr < 4; pr++) read_words(ring, 0, pr, raw[0]), read_words(ring, 1, pr, raw[1]);
    read_group(ring, 0, raw[0]);
#pragma unroll
    for (int i = 0; i < MT; i++) read_x(ring, 0, i, xa[0]);
    start_group(raw[0]);
#pragma unroll
    for (int pr = 0; pr < 4; pr++) unpack(raw[0], pr, op[0]);
    int slot = 0;
    auto stage_steps = [&](int kt, auto odd_c) __attribute__((always_inline)) {
        const int next = slot == NS - 1 ? 0 : slot + 1;
        const int younger = min(ns - 1, kt + NS - 1) - (kt + 1);
        const uint8_t *cur = ring + slot * C::STAGE_BYTES, *nxt = ring + next * C::STAGE_BYTES;
        if (C::BF && kt + 1 < ns) {
            wait_stage(younger, std::integral_constant<bool, !decltype(odd_c)::value>{});
            convert_read(next);
        }
        __builtin_amdgcn_sched_barrier(0);
        sub_step(I0{}, odd_c, cur, cur);
        if (C::BF && kt + 1 < ns) convert_write(next);
        sub_step(I1{}, odd_c, cur, cur);
#pragma unroll
        for (int i = 0; i < MT; i++) read_x(cur, 3, i, xa[1]);  // the last reads of the slot
        if (!C::BF) wait_stage(younger, std::integral_constant<bool, !decltype(odd_c)::value>{});
        lds_barrier();
        if (kt + NS < ns) issue(kt + NS, slot);
        __builtin_amdgcn_sched_barrier(0);
        sub_step(I2{}, odd_c, nxt, nullptr);
        sub_step(I3{}, odd_c, nxt, nxt);
        slot = next;
    };
#pragma unroll 1
    for (int kt = 0; kt < ns; kt += C::UNIT) {
        stage_steps(kt, std::false_type{});
        if constexpr (C::FOLD) stage_steps(kt + 1, std::true_type{});
    }
    for (int kt = ns; kt < n_block; kt++) lds_barrier();  // a slice with fewer stages than the block's longest
    if constexpr (C::FOLD) {
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int i = 0; i < MT; i++) fold_tile(p, i);
    }

    // ---- the slices add up in slice order; slice s finishes the quads s Q / KS .. of every lane
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // every wavefront is done reading the stages
    constexpr int QS = C::Q / KS;
    auto quad = [&](int q) __attribute__((always_inline)) {  // quad q: channel q / (4 MT), token tile (q / 4) % MT, tokens 8 (q % 4) + 4 khalf ..
        const int p = q / (4 * MT), i = (q / 4) % MT, r = 4 * (q & 3);
        const v16f& t = C::FOLD ? y[p][C::FOLD ? i : 0] : acc[p][i];
        return make_float4(t[r], t[r + 1], t[r + 2], t[r + 3]);
    };
    float4 mine[QS];
    if constexpr (KS > 1) {
        float4* red = reinterpret_cast<float4*>(smem);  // [owner][source, without the owner][QS][4 wavefronts][64]
#pragma unroll
        for (int o = 0; o < KS; o++)
            if (o != slice) {
                const int src = slice - (slice > o ? 1 : 0);
#pragma unroll
                for (int q = 0; q < QS; q++) red[((o * (KS - 1) + src) * QS + q) * 256 + wv * kWave + lane] = quad(o * QS + q);
            }
        __syncthreads();
#pragma unroll
        for (int o = 0; o < KS; o++)
            if (o == slice) {
#pragma unroll
                for (int q = 0; q < QS; q++) {
                    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                    for (int s = 0; s < KS; s++) {
                        const float4 t = s == o ? quad(o * QS + q) : red[((o * (KS - 1) + s - (s > o ? 1 : 0)) * QS + q) * 256 + wv * kWave + lane];
                        v = s == 0 ? t : make_float4(v.x + t.x, v.y + t.y, v.z + t.z, v.w + t.w);
                    }
                    mine[q] = v;
                }
            }
    } else {
#pragma unroll
        for (int q = 0; q < QS; q++) mine[q] = quad(q);
    }
    if (a.splits > 1) {  // block-uniform: whole accumulator blocks, in the order of the registers; awq_stream_finish_kernel adds and transposes them
        float4* dst = reinterpret_cast<float4*>(a.partials) + ((int64_t)(split * a.slabs + slab) * a.tiles_n + tile) * (C::Q * 256);
#pragma unroll
        for (int q = 0; q < QS; q++) dst[(slice * QS + q) * 256 + wv * kWave + lane] = mine[q];
        return;
    }
    float bias[2] = {0.f, 0.f};
    if (a.bias)
#pragma unroll
        for (int p = 0; p < 2; p++) bias[p] = Lo<LLMQ_F16>::to_f32(a.bias[min(8 * cw + channel_of(wv, p), a.N - 1)]);
    if constexpr (KS > 1) __syncthreads();  // the sums are read: the finished tile takes their place
#pragma unroll
    for (int q = 0; q < QS; q++) {
        const int qq = slice * QS + q, p = qq / (4 * MT), ch = 8 * l32 + channel_of(wv, p);
        const int row = 32 * ((qq / 4) % MT) + 8 * (qq & 3) + 4 * khalf;
        const float bv = p ? bias[1] : bias[0];
        const float v[4] = {mine[q].x, mine[q].y, mine[q].z, mine[q].w};
#pragma unroll
        for (int e = 0; e < 4; e++)
            *reinterpret_cast<uint16_t*>(smem + (row + e) * kOutStride + 2 * ch) = finish_value<C::BF>(v[e], a.bias != nullptr, bv);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < rows * kTileWords; i += C::NT) {
        const int row = i / kTileWords, c = i % kTileWords, ch = tile * kTileCh + 8 * c;
        if (ch < a.N) store_streaming(a.out + (int64_t)(m0 + row) * a.N + ch, *reinterpret_cast<const uint4*>(smem + row * kOutStride + 16 * c));
    }
}

// Adds the accumulator blocks of a K split in split order: a block of threads finishes 8 tokens x 256 channels.
template <int MT, bool BF>
__global__ __launch_bounds__(256) void awq_stream_finish_kernel(StreamArgs a) {
    constexpr int Q = 8 * MT;
    __shared__ __attribute__((aligned(16))) uint8_t tile_out[8 * kOutStride];
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave, l32 = lane & 31, khalf = lane >> 5;
    const int g = blockIdx.x % (4 * MT), tile = (blockIdx.x / (4 * MT)) % a.tiles_n, slab = blockIdx.x / (4 * MT) / a.tiles_n;
    const int m0 = slab * 32 * MT + 8 * g, rows = min(8, a.M - m0);
    if (rows <= 0) return;  // block-uniform, before any barrier
    const int64_t stride = (int64_t)a.slabs * a.tiles_n * (Q * 256);  // float4s between splits
    const float4* src = reinterpret_cast<const float4*>(a.partials) + ((int64_t)slab * a.tiles_n + tile) * (Q * 256) + wv * kWave + lane;
    float4 s0 = make_float4(0.f, 0.f, 0.f, 0.f), s1 = s0;
    constexpr int U = 4;
    for (int sp = 0; sp < a.splits; sp += U) {
        float4 t0[U], t1[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const float4* p = src + min(sp + u, a.splits - 1) * stride;
            t0[u] = p[g * 256];
            t1[u] = p[(4 * MT + g) * 256];
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (sp + u < a.splits) {
                s0 = make_float4(s0.x + t0[u].x, s0.y + t0[u].y, s0.z + t0[u].z, s0.w + t0[u].w);
                s1 = make_float4(s1.x + t1[u].x, s1.y + t1[u].y, s1.z + t1[u].z, s1.w + t1[u].w);
            }
    }
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const int ch = 8 * l32 + channel_of(wv, p);
        const float bv = a.bias ? Lo<LLMQ_F16>::to_f32(a.bias[min(tile * kTileCh + ch, a.N - 1)]) : 0.f;
        const float4 v4 = p ? s1 : s0;
        const float v[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
        for (int e = 0; e < 4; e++)
            *reinterpret_cast<uint16_t*>(tile_out + (4 * khalf + e) * kOutStride + 2 * ch) = finish_value<BF>(v[e], a.bias != nullptr, bv);
    }
    __syncthreads();
    const int row = threadIdx.x >> 5, c = threadIdx.x & 31, ch = tile * kTileCh + 8 * c;
    if (row < rows && ch < a.N) store_streaming(a.out + (int64_t)(m0 + row) * a.N + ch, *reinterpret_cast<const uint4*>(tile_out + row * kOutStride + 16 * c));
}

inline int cdiv_s(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }

template <class C>
int launch_cfg(const StreamArgs& a, hipStream_t st) {
    auto kernel = awq_stream_kernel<C>;
    // per device: the attribute belongs to the loaded code object of the current device
    static bool raised[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return LLMQ_ERR_LAUNCH;
    if (dev < 0 || dev >= 64 || !raised[dev]) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES) != hipSuccess)
            return LLMQ_ERR_LAUNCH;
        if (dev >= 0 && dev < 64) raised[dev] = true;
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)(a.tiles_n * a.splits * a.slabs)), dim3(C::NT), C::LDS_BYTES, st, a);
    if (a.splits > 1)
        hipLaunchKernelGGL((awq_stream_finish_kernel<C::MT, C::BF>), dim3((unsigned)(4 * C::MT * a.tiles_n * a.slabs)), dim3(256), 0, st, a);
    return launch_status();
}
template <bool BF, int V>
int launch_variant(int cfg, bool fold, const StreamArgs& a, hipStream_t st) {
    switch (cfg) {
        case 0: return fold ? launch_cfg<StreamCfg<1, 2, 4, true, BF, V>>(a, st) : launch_cfg<StreamCfg<1, 2, 4, false, BF, V>>(a, st);
        case 1: return fold ? launch_cfg<StreamCfg<2, 2, 4, true, BF, V>>(a, st) : launch_cfg<StreamCfg<2, 2, 4, false, BF, V>>(a, st);
        case 2: return fold ? launch_cfg<StreamCfg<2, 1, 4, true, BF, V>>(a, st) : launch_cfg<StreamCfg<2, 1, 4, false, BF, V>>(a, st);
        case 3: return launch_cfg<StreamCfg<4, 2, 3, false, BF, V>>(a, st);
        default: return launch_cfg<StreamCfg<4, 1, 3, false, BF, V>>(a, st);
    }
}

// Configurations: 32-token tiles per block and K slices; their cost by FOLD (us): `step` per stage of a slice, of which a share 1 - lo goes with the
// fraction of the CUs that is busy (the chip is power-managed, and the blocks share the supply), `fixed` per round of blocks, `first`: with
// two slices (a block fills a CU) once per launch, with one slice (two blocks fit a CU) the share of a block's time that one beside it adds.
// Fitted on an MI355X to every configuration x K split of 900 random problems of up to 2048 tokens (22 000 plans; groups of 32, 64, 128; weights out
// of HBM), for the time of the plan it picks: 0.9 % behind the best plan in the mean.  Besides: MB of weights and outputs, and for a K split the
// finishing launch and its MB of partial sums.
struct StreamCost { double step, lo, fixed, first; };
struct StreamShape { int mt, ks; StreamCost cost[2]; };  // cost: without / with FOLD
const StreamShape kStream[kAwqStreamConfigs] = {
    {1, 2, {{1.032, 0.750, 3.698, 1.320}, {0.765, 0.785, 4.363, 1.287}}},
    {2, 2, {{1.193, 0.836, 2.873, 1.935}, {0.949, 0.906, 4.591, 1.275}}},
    {2, 1, {{0.673, 1.294, 4.190, 0.872}, {0.571, 1.131, 4.957, 0.651}}},
    {4, 2, {{1.348, 0.998, 4.101, 1.354}, {0, 0, 0, 0}}},
    {4, 1, {{0.699, 1.336, 4.996, 0.851}, {0, 0, 0, 0}}}};
constexpr double kWeightsUs = 0.129, kWeightsBase = 4.67, kOutUs = 0.336, kFinishUs = 1.86, kPartialUs = 0.424;

size_t partials_of(const AwqStreamPlan& p, int64_t M, int64_t N) {
    const int mt = kStream[p.cfg].mt;
    return p.splits > 1 ? (size_t)p.splits * cdiv_s(M, 32 * mt) * cdiv_s(N, kTileCh) * (32 * mt * kTileCh * 4) : 0;
}
AwqStreamPlan plan_of(int cfg, bool fold, int64_t K, int splits) {
    const int ks = kStream[cfg].ks, units = (int)(K / (kStageK * (fold ? 2 : 1)));
    AwqStreamPlan p{cfg, fold ? 1 : 0, 1, cdiv_s(cdiv_s(units, splits), ks) * ks};  // equal shares for the slices
    p.splits = cdiv_s(units, p.units_per_block);
    return p;
}
double time_of(const AwqStreamPlan& p, int64_t M, int64_t N, int64_t K) {
    const StreamShape& c = kStream[p.cfg];
    const StreamCost& q = c.cost[p.fold];
    const double x = (double)cdiv_s(N, kTileCh) * cdiv_s(M, 32 * c.mt) * p.splits / 256, full = std::floor(x), part = x - full;
    const double run = p.units_per_block * (p.fold ? 2 : 1) / (double)c.ks * q.step;
    double t;
    if (c.ks == 2) t = full * (run + q.fixed) + (part > 0 ? run * (q.lo + (1 - q.lo) * part) + q.fixed : 0) + q.first;
    else t = run * (x > 1 ? std::max(x, 1 + (std::ceil(x) - 1) * q.first) : q.lo + (1 - q.lo) * x) + q.fixed * std::max(1.0, std::ceil(x / 2));
    const double w = (double)N * K * 0.5e-6 * kWeightsUs + kWeightsBase, t3 = t * t * t, w3 = w * w * w;
    double rest = kOutUs * 2e-6 * (double)M * N;
    if (p.splits > 1) rest += kFinishUs + kPartialUs * 1e-6 * (double)partials_of(p, M, N);
    return std::cbrt(std::sqrt(t3 * t3 + w3 * w3)) + rest;
}

}  // namespace

// K in whole stages; 32-bit byte offsets into a stage, the scales and the zero points; group numbers by a 32-bit reciprocal
bool awq_stream_supported(int64_t M, int64_t N, int64_t K, int64_t group, int64_t ldx) {
    return M >= 1 && M <= (1 << 24) && N >= 8 && N <= (1 << 24) && K >= kStageK && K % kStageK == 0 && K <= (1 << 20) && group >= 32 && group % 32 == 0 && K % group == 0 &&
           ldx < (1 << 22) && (K / group) * N < ((int64_t)1 << 30) && (int64_t)cdiv_s(N, kTileCh) * cdiv_s(M, 32) <= (1 << 24);
}

// The plan of a problem among those whose partial sums take at most `max_partials` bytes (a plan without a K split always does).
// Up to 64 tokens a group that is a multiple of 128 keeps its exact integers (FOLD); beyond, where the tile kernel rounded every weight, either.
AwqStreamPlan make_awq_stream_plan(int64_t M, int64_t N, int64_t K, int64_t group, size_t max_partials, int force_cfg, int force_splits) {
    const bool foldable = group % 128 == 0;
    AwqStreamPlan best{};
    double best_t = 1e300;
    for (int cfg = 0; cfg < kAwqStreamConfigs; cfg++) {
        const int mt = kStream[cfg].mt;
        if (force_cfg >= 0 ? cfg != force_cfg : (mt == 1 && M > 64) || (mt == 2 && M <= 16) || (mt == 4 && M <= 64)) continue;
        const bool fold = foldable && mt <= 2;
        for (int sp = 1; sp <= 24; sp += sp < 8 ? 1 : sp < 16 ? 2 : 4) {
            const AwqStreamPlan p = plan_of(cfg, fold, K, force_splits > 0 ? force_splits : sp);
            const int64_t blocks = (int64_t)cdiv_s(N, kTileCh) * cdiv_s(M, 32 * mt) * p.splits;
            if (p.splits > 1 && (partials_of(p, M, N) > max_partials || (force_splits <= 0 && (blocks > 640 || partials_of(p, M, N) > (size_t)300 << 20)))) {
                if (force_splits <= 0) break;
                return plan_of(cfg, fold, K, 1);
            }
            if (force_splits > 0) return p;
            double t = time_of(p, M, N, K);
            // Past 64 tokens with few weights and a short K a K split of two 64-token blocks a CU comes out cheaper than the table has it, most where the
            // alternative is one launch over eight to twelve stages (us, one launch / split: 148 x 632 x 512 10.0 / 8.5, 79 x 1560 x 512 10.0 / 8.7).
            // 1200 random problems of 65-600 tokens and up to 4 million weights, against the tile kernel: more than 8 % behind 62 -> 18, more than 3 %
            // 266 -> 187, in the mean 1.07 -> 1.08 times ahead.  With a longer K such a split loses 2-6 % (391 x 512 x 2432 13.3 / 14.3).
            if (cfg == 2 && p.splits > 1 && M > 64 && K <= 1024 && N * K <= 4000000) t -= 0.9;
            if (t < best_t) best_t = t, best = p;
        }
    }
    return best;
}

size_t awq_stream_workspace_bytes(const AwqStreamPlan& p, int64_t M, int64_t N) { return partials_of(p, M, N); }

int launch_awq_stream(const AwqStreamPlan& p, const uint16_t* x, int64_t ldx, const uint32_t* qw, const uint16_t* scales, const uint32_t* qz,
                      const uint16_t* bias, uint16_t* out, float* ws, int M, int N, int K, int G, bool bf16_io, hipStream_t st) {
    const uint32_t hpg = (uint32_t)G / 32u;
    const StreamArgs a{x, qw, scales, qz, bias, out, ws, ldx, M, N, K, (int)hpg, (uint32_t)((((uint64_t)1 << 32) + hpg - 1) / hpg), p.units_per_block,
                       cdiv_s(N, kTileCh), p.splits, cdiv_s(M, 32 * kStream[p.cfg].mt)};
    const bool whole = N % 32 == 0;  // rows of packed words are whole 16-byte pieces
    if (bf16_io) return whole ? launch_variant<true, 4>(p.cfg, p.fold, a, st) : launch_variant<true, 1>(p.cfg, p.fold, a, st);
    return whole ? launch_variant<false, 4>(p.cfg, p.fold, a, st) : launch_variant<false, 1>(p.cfg, p.fold, a, st);
}

}  // namespace llmq
