// W8A8 int8 / FP8 GEMM for a decode batch: up to 64 tokens, weight rows streamed through LDS in long pieces.
//
//   acc[m,n] = sum_k A[m,k] * B[n,k]        A: [M,K] row-major, B: [N,K] row-major (both K-contiguous)
//
// What bounds it is the stream of weights out of HBM, and how fast that runs depends on how long a piece of a row is asked for at once
// (weights only, 37888 x 3584 bytes: 128 rows x 128 bytes per block and step 28.6 us, 16 rows x 512 bytes 22.6 us = 6.0 TB/s).
// Operands that go straight into registers (gemm_skinny.hip) fetch 64 or 128 bytes of a row per load, and the 64 and 32 KB stages of the tile
// kernel 128 bytes.  So here
//   * a block of four wavefronts owns 16 T channels and up to 16 MT tokens over the whole K: no K split, no partial sums, no second launch;
//   * a stage is SEG = 512 or 1024 bytes of K of each weight row and each activation row, loaded straight into LDS; NS - 1 stages are in
//     flight while one is multiplied, and the wait is for the oldest only;
//   * each wavefront multiplies its quarter of the bytes of each stage and the block adds the four sums in wavefront order at the end.
// The activations are re-read by every block out of the L2: T = 2 and 4 halve and quarter that for many channels, T = 1 makes more blocks.
// MANY: for many channels a block that ends with its channels leaves the CU without loads while the next one starts, which costs a quarter of the
// stream (37888 channels: 592 blocks of 64).  There as many blocks as are resident take one group of channels after the other: the ring
// runs on into the next group while the last one's sums are added beside it, and the scales of all groups are in LDS from the start, so that the
// epilogue waits for no load.  (For 17-32 tokens, with twice the activations per stage, level with the tiles: 32 x 37888 x 3584 31.7 / 32.8 us,
// 32 x 30000 x 2048 16.3 / 13.5; not kept.)
// 1024-byte pieces are for few blocks over a long K (K = 18944 at N = 3584: 512 bytes 3.0 TB/s, 1024 bytes 4.2 TB/s).
//
// Measured (int8, weights out of HBM, us; before: the fastest plan of skinny and tile kernels the planner had):
//   tokens        16 x 4608 x 3584   16 x 3584 x 3584   16 x 896 x 4864   16 x 3584 x 18944   32 x 4608 x 3584   64 x 3584 x 3584
//   before              9.9                7.1                9.4               19.4               11.4               12.3
//   this kernel         6.8                5.7                5.5               16.0                8.0                8.2
// MANY, before / now:  1 x 37888 x 3584 30.9 / 25.0 (5.4 TB/s with launch and tail), 16 x 37888 x 3584 32.4 / 27.2, 8 x 11904 x 8192 24.9 / 19.7.
#include <algorithm>
#include <type_traits>

#include "gemm_rows.h"

namespace llmq {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

constexpr int kRowsGroups = 16;  // groups of channels a block takes at most

template <bool FP8_, int AFMT_, int T_, int MT_, int SEG_, int NS_, bool MANY_ = false>
struct RowsCfg {
    static constexpr bool FP8 = FP8_;
    static constexpr int AFMT = AFMT_;
    static constexpr int T = T_, MT = MT_;              // 16-channel / 16-token tiles of a block
    static constexpr int SEG = SEG_, NS = NS_;          // bytes of a row per stage; LDS stages
    static constexpr int NW = 4, NT = NW * kWave;
    static constexpr int CPR = SEG / 16;                // 16-byte chunks of a row
    static constexpr int KSTEP = FP8 ? 128 : 64;        // K-bytes of an MFMA
    static constexpr int STEPS = SEG / NW / KSTEP;      // MFMA steps of a wavefront per stage
    static constexpr int ROWS = 16 * (T + MT), STAGE_BYTES = ROWS * SEG;
    static constexpr int LPT = STAGE_BYTES / (NT * 16);  // direct loads per thread and stage
    static constexpr bool MANY = MANY_;                 // a block takes several groups of channels, one after the other
    static constexpr int RING_BYTES = NS * STAGE_BYTES, SUM_BYTES = NW * T * MT * kWave * 16;
    // MANY: the ring stays in flight while the wavefronts add up, beside it, and the scales of all groups lie behind that
    static constexpr int LDS_BYTES = RING_BYTES + (MANY ? SUM_BYTES + (kRowsGroups * 16 * T * 2 + 16 * MT) * 4 : 0);
    static_assert(STEPS >= 1 && SEG % (NW * KSTEP) == 0 && STAGE_BYTES % (NT * 16) == 0, "a stage splits evenly");
    static_assert(LDS_BYTES <= 160 * 1024 && (NS - 1) * LPT < 64 && RING_BYTES >= SUM_BYTES, "LDS, vmcnt, the final sum");
};

template <class C>
__global__ __launch_bounds__(C::NT) void gemm_rows_kernel(const uint8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb,
                                                          int M, int N, int K, SkinnyEpilogue ep, void* __restrict__ out, int64_t ldo,
                                                          void* __restrict__ acc_dump) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr int T = C::T, MT = C::MT, NS = C::NS, SEG = C::SEG;
    using acc_t = typename std::conditional<C::FP8, v4f, v4i>::type;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int r16 = lane & 15, kq = lane >> 4;
    int n0 = blockIdx.x * (16 * T);
    const int nst = (K + SEG - 1) / SEG, step_n = C::MANY ? gridDim.x * (16 * T) : 0;
    const int mine = C::MANY ? (N - n0 + step_n - 1) / step_n : 1, total = mine * nst;  // groups and stages of the block

    // ---- direct loads: piece p of a stage is row p / CPR (weights, then activations), LDS chunk p % CPR, which holds chunk
    // (p % CPR) ^ (row & 15) of the row, so that the operand reads of 16 rows hit 16 places
    const uint8_t* wb = B + (int64_t)n0 * ldb;
    uint32_t off[C::LPT], chunk[C::LPT];
#pragma unroll
    for (int i = 0; i < C::LPT; i++) {
        const int p = (wave * C::LPT + i) * kWave + lane, row = p / C::CPR;
        chunk[i] = 16u * (uint32_t)((p % C::CPR) ^ (row & 15));
        off[i] = row < 16 * T ? (uint32_t)min(row, N - 1 - n0) * (uint32_t)ldb : (uint32_t)min(row - 16 * T, M - 1) * (uint32_t)lda;
    }
    int issue_n0 = n0;
    auto next_group = [&]() __attribute__((always_inline)) {  // of the loads
        issue_n0 += step_n;
        wb = B + (int64_t)issue_n0 * ldb;
        if (issue_n0 + 16 * T <= N) return;
#pragma unroll
        for (int i = 0; i < C::LPT; i++) {
            const int row = ((wave * C::LPT + i) * kWave + lane) / C::CPR;
            if (row < 16 * T) off[i] = (uint32_t)min(row, N - 1 - issue_n0) * (uint32_t)ldb;
        }
    };
    const uint32_t lds_base = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)smem);
    auto issue = [&](int s, int slot) __attribute__((always_inline)) {
        const bool tail = (s + 1) * SEG > K;  // uniform: chunks past the end re-read the last one of the row, masked when used
#pragma unroll
        for (int i = 0; i < C::LPT; i++) {
            const bool w = (wave * C::LPT + i) * kWave < 16 * T * C::CPR;  // wavefront-uniform
            const uint8_t* src = (w ? wb : A) + (int64_t)s * SEG;
            uint32_t voff = off[i] + chunk[i];
            if (tail) voff = off[i] + min(chunk[i], (uint32_t)(K - 16 - s * SEG));
            const uint32_t m0v = lds_base + (uint32_t)(slot * C::STAGE_BYTES + (wave * C::LPT + i) * 1024);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0v), "v"(voff), "s"(src) : "memory", "m0");
        }
    };
    auto lds_barrier = []() __attribute__((always_inline)) {  // orders LDS traffic only: the loads stay in flight across it
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    acc_t acc[MT][T];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int t = 0; t < T; t++) acc[mt][t] = acc_t{0, 0, 0, 0};

    using frag_t = typename std::conditional<C::FP8, v8i, v4i>::type;
    auto read = [&](const uint8_t* st, int row, int step, bool tail, int left) __attribute__((always_inline)) {  // row of the stage
        const u4* r = reinterpret_cast<const u4*>(st + row * SEG);
        if constexpr (C::FP8) {
            const int c = (wave * C::STEPS + step) * 8 + 2 * kq;
            u4 lo = r[c ^ r16], hi = r[(c + 1) ^ r16];
            if (tail) {
                if (16 * c >= left) lo = u4{0, 0, 0, 0};
                if (16 * (c + 1) >= left) hi = u4{0, 0, 0, 0};
            }
            return v8i{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
        } else {
            const int c = (wave * C::STEPS + step) * 4 + kq;
            u4 v = r[c ^ r16];
            if (tail && 16 * c >= left) v = u4{0, 0, 0, 0};
            return v4i{(int)v[0], (int)v[1], (int)v[2], (int)v[3]};
        }
    };
    auto compute = [&](int slot, bool tail, int left) __attribute__((always_inline)) {
        const uint8_t* st = smem + slot * C::STAGE_BYTES;
#pragma unroll
        for (int step = 0; step < C::STEPS; step++) {
            frag_t b[T], a[MT];
#pragma unroll
            for (int t = 0; t < T; t++) b[t] = read(st, 16 * t + r16, step, tail, left);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) a[mt] = read(st, 16 * (T + mt) + r16, step, tail, left);
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int t = 0; t < T; t++) {
                    if constexpr (C::FP8) acc[mt][t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b[t], a[mt], acc[mt][t], 0, C::AFMT, 0, 0, 0, 0);
                    else acc[mt][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b[t], a[mt], acc[mt][t], 0, 0, 0);
                }
        }
    };
    auto wait_stage = [&](int younger) __attribute__((always_inline)) {  // the oldest stage in flight has landed when `younger` later ones remain
#define LLMQ_ROWS_WAIT(Y) \
    if (NS - 1 > (Y) && younger == (Y)) { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(((Y) < NS ? (Y) : 0) * C::LPT) : "memory"); return; }
        LLMQ_ROWS_WAIT(6) LLMQ_ROWS_WAIT(5) LLMQ_ROWS_WAIT(4) LLMQ_ROWS_WAIT(3) LLMQ_ROWS_WAIT(2) LLMQ_ROWS_WAIT(1)
#undef LLMQ_ROWS_WAIT
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    static_assert(NS <= 8, "wait_stage");

    // scales and bias of channel n0 + c of group g: MANY keeps those of all its groups in LDS, so that no load of the epilogue waits behind the ring
    float* s_w = reinterpret_cast<float*>(smem + C::RING_BYTES + C::SUM_BYTES);
    float* s_b = s_w + kRowsGroups * 16 * T;
    float* s_a = s_b + kRowsGroups * 16 * T;
    const float alpha = ep.alpha * (ep.alpha_dev ? *ep.alpha_dev : 1.0f);
    const float out_scale = ep.out_scale ? *ep.out_scale : 1.f;
    auto weight_scale = [&](int n) __attribute__((always_inline)) { return ep.w_scale ? ep.w_scale[min(n, N - 1)] : 1.f; };
    auto bias_of = [&](int n) __attribute__((always_inline)) { return ep.bias ? ep.beta * load_as_f32(ep.bias, ep.bias_dtype, min(n, N - 1)) : 0.f; };
    if constexpr (C::MANY) {
        for (int i = tid; i < mine * 16 * T; i += C::NT) {
            const int n = n0 + i / (16 * T) * step_n + i % (16 * T);
            s_w[i] = weight_scale(n), s_b[i] = bias_of(n);
        }
        if (tid < 16 * MT) s_a[tid] = ep.a_scale ? ep.a_scale[min(tid, M - 1)] : 1.f;
    }

    // ---- the wavefronts add up in wavefront order, then scales, bias, store
    acc_t (*red)[MT * T][kWave] = reinterpret_cast<acc_t (*)[MT * T][kWave]>(smem + (C::MANY ? C::RING_BYTES : 0));
    auto finish = [&](int group) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int t = 0; t < T; t++) red[wave][mt * T + t][lane] = acc[mt][t];
        lds_barrier();
        for (int idx = tid; idx < MT * T * kWave; idx += C::NT) {
            const int q = idx / kWave, l = idx % kWave, mt = q / T, t = q % T;
            acc_t sum = red[0][q][l];
#pragma unroll
            for (int w = 1; w < C::NW; w++) sum += red[w][q][l];
            // lane l of that accumulator: token 16 mt + l % 16, channels n0 + 16 t + 4 (l / 16) .. + 3
            const int m = 16 * mt + (l & 15), c = 16 * t + 4 * (l >> 4), n = n0 + c;
            if (m >= M || n >= N) continue;
            const float sa = C::MANY ? s_a[m] : ep.a_scale ? ep.a_scale[m] : 1.f;
            uint16_t h[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float sw = C::MANY ? s_w[group * 16 * T + c + e] : weight_scale(n + e);
                const float bb = C::MANY ? s_b[group * 16 * T + c + e] : bias_of(n + e);
                const float v = epi_value((float)sum[e], sa, sw, alpha, bb);
                h[e] = ep.out_dtype == LLMQ_BF16 ? Lo<LLMQ_BF16>::from_f32(v) : Lo<LLMQ_F16>::from_f32(v);
            }
            uint16_t* orow = reinterpret_cast<uint16_t*>(out) + (int64_t)m * ldo + n;
            if (ep.out_scale) {
                float* frow = reinterpret_cast<float*>(out) + (int64_t)m * ldo + n;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float f = ep.out_dtype == LLMQ_BF16 ? Lo<LLMQ_BF16>::to_f32(h[e]) : Lo<LLMQ_F16>::to_f32(h[e]);
                    if (n + e < N) frow[e] = fp8_round_trip(f, out_scale);
                }
            } else if (n + 3 < N && ((reinterpret_cast<uintptr_t>(orow) & 7u) == 0)) {
                *reinterpret_cast<uint2*>(orow) = make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < N) orow[e] = h[e];
            }
            if (acc_dump) {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < N) {
                        const auto sv = sum[e];  // scalar copy first: a bit cast applied to the vector element itself reads element 0
                        reinterpret_cast<uint32_t*>(acc_dump)[(int64_t)m * N + n + e] = __builtin_bit_cast(uint32_t, sv);
                    }
            }
        }
    };

    int issued = 0, issue_s = 0;  // stages in flight or done; the next one within its group
    auto issue_next = [&](int slot) __attribute__((always_inline)) {
        if (issued == total) return;
        if (C::MANY && issue_s == nst) issue_s = 0, next_group();
        issue(issue_s++, slot);
        issued++;
    };
#pragma unroll
    for (int t = 0; t < NS - 1; t++) issue_next(t);
    int slot = 0, s = 0, group = 0;
#pragma unroll 1
    for (int f = 0; f < total; f++) {
        wait_stage(min(total - 1, f + NS - 2) - f);
        lds_barrier();  // publishes this stage; every wavefront has read the whole of the one before
        issue_next(slot == 0 ? NS - 1 : slot - 1);
        if ((s + 1) * SEG > K) compute(slot, true, K - s * SEG);
        else compute(slot, false, 0);
        slot = slot == NS - 1 ? 0 : slot + 1;
        if (C::MANY && ++s == nst) {
            finish(group);  // its reads of the sums are done in every wavefront before the barrier of the next stage
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int t = 0; t < T; t++) acc[mt][t] = acc_t{0, 0, 0, 0};
            n0 += step_n, group++, s = 0;
        } else if (!C::MANY) s++;
    }
    if constexpr (!C::MANY) {
        lds_barrier();  // every wavefront is done reading the stages
        finish(0);
    }
}

template <class C>
int launch_rows(const uint8_t* A, int64_t lda, const uint8_t* B, int64_t ldb, int M, int N, int K, const SkinnyEpilogue& ep, void* out, int64_t ldo,
                void* acc_dump, hipStream_t st) {
    auto kernel = gemm_rows_kernel<C>;
    if (C::LDS_BYTES > 64 * 1024) {
        // per device: the attribute belongs to the loaded code object of the current device
        static bool raised[64] = {};
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return LLMQ_ERR_LAUNCH;
        if (dev < 0 || dev >= 64 || !raised[dev]) {
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES) != hipSuccess)
                return LLMQ_ERR_LAUNCH;
            if (dev >= 0 && dev < 64) raised[dev] = true;
        }
    }
    int blocks = (N + 16 * C::T - 1) / (16 * C::T);
    if (C::MANY) {  // as many as are resident at once, or fewer so that all take as many groups (288 groups of 18432 x 11904: 144 blocks 43.6 us, 256 52.7)
        const int slots = 256 * (160 * 1024 / C::LDS_BYTES), each = std::min(kRowsGroups, (blocks + slots - 1) / slots);
        blocks = (blocks + each - 1) / each;
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(C::NT), C::LDS_BYTES, st, A, lda, B, ldb, M, N, K, ep, out, ldo,
                       acc_dump);
    return launch_status();
}

template <bool FP8, int AFMT>
int launch_variant(int variant, const uint8_t* A, int64_t lda, const uint8_t* B, int64_t ldb, int M, int N, int K, const SkinnyEpilogue& ep, void* out,
                   int64_t ldo, void* acc_dump, hipStream_t st) {
    switch (variant) {
#define LLMQ_ROWS_CASE(I, T, MT, SEG, NS, MANY) \
    case I: return launch_rows<RowsCfg<FP8, AFMT, T, MT, SEG, NS, MANY>>(A, lda, B, ldb, M, N, K, ep, out, ldo, acc_dump, st);
        LLMQ_ROWS_VARIANTS(LLMQ_ROWS_CASE)
#undef LLMQ_ROWS_CASE
    }
    return LLMQ_ERR_SHAPE;
}

}  // namespace

int launch_gemm_rows(bool fp8, int a_format, int variant, const uint8_t* A, int64_t lda, const uint8_t* B, int64_t ldb, int M, int N, int K,
                     const SkinnyEpilogue& ep, void* out, int64_t ldo, void* acc_dump, hipStream_t st) {
    if (variant < 0 || variant >= kRowsVariants || M > 16 * kRowsShapes[variant].mt) return LLMQ_ERR_SHAPE;
    if (!fp8) return launch_variant<false, 0>(variant, A, lda, B, ldb, M, N, K, ep, out, ldo, acc_dump, st);
    if (a_format == 0) return launch_variant<true, 0>(variant, A, lda, B, ldb, M, N, K, ep, out, ldo, acc_dump, st);
    return launch_variant<true, 1>(variant, A, lda, B, ldb, M, N, K, ep, out, ldo, acc_dump, st);
}

}  // namespace llmq
