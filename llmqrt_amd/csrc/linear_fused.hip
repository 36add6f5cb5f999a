// Few-token quantized linear in one launch: activation quantizer (dynamic per token, dynamic per tensor, or static) + W8A8 int8 /
// FP8 GEMM + dequant epilogue, for up to 16 tokens (decode).
//
//   s[m]    = round_dt( max(absmax_k |x[m,k]|, round_dt(floor)) / qmax )            the row quantizers of quant.hip
//   q[m,k]  = narrow( clamp( round_dt( x[m,k] / s[m] ) ) )
//   out     = ((sum_k q[m,k] * B[n,k]) * s[m]) * sw[n] + bias[n]                     llmq_gemm_w8a8 / llmq_gemm_fp8
//
// The reference runs these as separate steps (nn_models/modules/linear/linear_sq.py:97-138: the quantizers of
// lines 44-65, then the GEMM op; linear_fp8.py:11-63 + 199-221, 296-311).  With a few tokens each step is a launch of a
// few microseconds that mostly waits; here the GEMM kernel quantizes its own activation operand:
//   * a wavefront owns 16*T output channels and one of NW consecutive runs of K steps, and the weights stream
//     from global memory straight into MFMA operand registers, exactly as in gemm_skinny.hip; a block has NG such sets of NW;
//   * before its first step a block quantizes the activations itself, once, into LDS, with all its wavefronts and NI more that do nothing
//     else: the codes as the [token][K] int8 / fp8 matrix the MFMA operand reads expect (the activations are a few KB per token and sit in
//     L2; every block repeats this, which is cheaper than a launch).  The first batch of weight loads is already in flight meanwhile;
//   * the arithmetic is the row quantizer's (quant_math.h), so codes and scales are bit-identical to llmq_quant_*, and so is
//     the result where the few-token GEMM splits K over as many wavefronts (int32 sums always; fp32 sums are else added in another order).
//
// What bounds it is a chain: launch, activation loads, maximum, codes, barrier, the operand reads of a few steps, the sum over the
// wavefronts.  A block of four wavefronts spent more time on its codes (14336 of them: 56 a lane, 10 instructions each) than on anything
// else, so up to 4096 channels, where a CU has one block at most, twelve more wavefronts help (int8 / fp8, us, four wavefronts / sixteen of
// which four multiply: 16 x 1152 x 896 6.2 / 5.5, 8 x 2304 x 2048 6.5 / 6.0, 16 x 896 x 4864 (two launches 13.7) - / 12.1).  With
// more channels the blocks of a CU would repeat the quantizer, so a block takes as many wavefronts as its codes need and 16 or 32
// channels (2 x 8448 x 1152 9.1 with two tiles a wavefront / 7.3, 7 x 15872 x 3840 two launches 24.1 / 16.8, 14336 codes: 16 x 9728 x 896 10.0 / 9.0).
// Lines between one launch and two: llmq_linear_one_launch_preferred and _ahead below.
#include <algorithm>
#include <type_traits>

#include "llmq_common.h"
#include "quant_math.h"

namespace llmq {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

struct FusedArgs {
    const uint16_t* x;       // [M, K] activations, row stride ldx elements
    const uint8_t* B;        // [N, K] quantized weights, row stride ldb bytes
    const float* w_scale;    // [N] or null
    const void* bias;        // [N] or null
    void* out;               // [M, N]
    uint8_t* q_dump;         // [M, K] quantized activations, or null
    float* scale_dump;       // [M] activation scales, or null
    void* acc_dump;          // [M, N] raw accumulators, or null
    int64_t ldx, ldb, ldo;
    int M, N, K;
    int bias_dtype, out_dtype;
    const float* in_scale;   // static: the activations' scale
    const float* out_scale;  // device scalar or null: out is fp32 and holds the value after a round trip through e4m3fn on it
};
// where the activation scale comes from: every row, the whole tensor, the caller
enum { SRC_TOKEN = 0, SRC_TENSOR = 1, SRC_STATIC = 2 };

constexpr int kRowPad = 16;        // bytes between LDS rows beyond K: consecutive tokens start 4 banks apart
constexpr int kMaxLdsBytes = 65536 - 256;  // llmq_linear_*_dynamic; llmq_linear_one_launch takes more of the CU's 160 KB
constexpr int kRowChunks = 10;     // 16-byte pieces of a row a lane keeps in registers (K <= 10 * 64 * 8 = 5120); longer rows are re-read

// NG sets of NW wavefronts along K, NI that only quantize; SRC_TENSOR, SRC_STATIC: CH 16-byte pieces of the tensor in a thread's registers
template <bool FP8, int DT, int T, int NW, int NG, int NI, int D, int SRC, int CH>
__global__ __launch_bounds__((NW * NG + NI) * kWave) void linear_fused_kernel(FusedArgs a) {
    constexpr bool TENSOR = SRC != SRC_TOKEN;  // one scale for the tensor
    constexpr int MODE = FP8 ? MODE_F8 : MODE_I8;
    constexpr int NWT = NW * NG + NI, NT = NWT * kWave, KSTEP = FP8 ? 128 : 64, P = FP8 ? 2 : 1, LB = 16 * P;  // LB codes per lane and step
    using acc_t = typename std::conditional<FP8, v4f, v4i>::type;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];  // [M][K + kRowPad] codes; after the main loop: red[NG * NW][T][64]
    __shared__ float s_scale[16];  // TENSOR: [0] = activation scale x weight scale
    __shared__ float s_red[TENSOR ? NWT : 1];

    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int r16 = lane & 15, kq = lane >> 4;
    const int M = a.M, N = a.N, K = a.K;
    const int kw = wave % NW, ng = wave / NW;  // run of K steps, set (NG and more: quantizes only)
    const int n0 = (blockIdx.x * NG + min(ng, NG - 1)) * (16 * T);
    const int steps = (K + KSTEP - 1) / KSTEP, spw = (steps + NW - 1) / NW;
    const int s_begin = ng < NG ? min(steps, kw * spw) : 0, s_end = ng < NG ? min(steps, s_begin + spw) : 0;
    const int row_bytes = K + kRowPad;

    const uint8_t* pb[T];
#pragma unroll
    for (int t = 0; t < T; t++) pb[t] = a.B + (int64_t)min(n0 + 16 * t + r16, N - 1) * a.ldb + kq * LB;

    struct Batch { u4 b[D][T][P]; };
    // K % 16 == 0: a lane's 16-byte pieces are either inside K or past it; a piece past the end re-reads the row's
    // first bytes and is masked when it is used
    auto load_batch = [&](int s0, Batch& d) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < D; i++) {
            const int s = min(s0 + i, s_end - 1);
#pragma unroll
            for (int p = 0; p < P; p++) {
                const int koff = s * KSTEP + kq * LB + 16 * p;
                const int kc = koff < K ? s * KSTEP + 16 * p : -(kq * LB);
#pragma unroll
                for (int t = 0; t < T; t++) d.b[i][t][p] = *reinterpret_cast<const u4*>(pb[t] + kc);
            }
        }
    };

    Batch ba, bb;
    // TENSOR: the activations are requested first (loads complete in order: behind the weights they would wait for HBM)
    uint4 act[CH];
    if constexpr (TENSOR) {
        const int cpr = K >> 3, total = M * cpr;
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const int i = min(tid + c * NT, total - 1), m = i / cpr;  // past the end: the last piece, which changes no maximum
            act[c] = reinterpret_cast<const uint4*>(a.x + (int64_t)m * a.ldx)[i - m * cpr];
        }
    }
    if (s_begin < s_end) load_batch(s_begin, ba);  // weights start streaming before the activations are quantized
    if constexpr (TENSOR) {
        const int cpr = K >> 3, total = M * cpr;
        float s;
        bool fin = false;  // block-uniform: the absmax behind the scale is finite, so no quotient can be NaN
        if constexpr (SRC == SRC_STATIC) {
            s = a.in_scale[0];
        } else {
            float amax = 0.f;
#pragma unroll
            for (int c = 0; c < CH; c++) amax = max_nonneg(amax, absmax8(act[c], DT == LLMQ_BF16));
            amax = block_max<NWT>(amax, s_red);
            s = scale_from_amax<DT, MODE>(amax);
            fin = amax < __builtin_inff() && s > 0.f;  // (the fp8 floor rounds to 0 in fp16: an all-zero tensor has scale 0 and 0 / 0)
        }
        const float inv_s = 1.0f / s;
        if (tid == 0) {
            const float alpha = s * a.w_scale[0];
            s_scale[0] = FP8 ? alpha : Lo<DT>::round(alpha);  // int8: rounded to the activation dtype, as store_alpha does
        }
        auto codes = [&](auto quot_c, auto fin_c) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < CH; c++) {
                const int i = tid + c * NT, m = i / cpr;
                if (i < total)
                    *reinterpret_cast<uint2*>(smem + m * row_bytes + 8 * (i - m * cpr)) =
                        quant8<DT, MODE, decltype(quot_c)::value, decltype(fin_c)::value>(act[c], s, inv_s);
            }
        };
        if constexpr (SRC == SRC_STATIC) {
            if (near_scale(s)) codes(std::integral_constant<int, Q_NEAR_F32>{}, std::false_type{});
            else codes(std::integral_constant<int, Q_DIV_F32>{}, std::false_type{});
        } else if (fin) codes(std::integral_constant<int, Q_DT>{}, std::true_type{});
        else codes(std::integral_constant<int, Q_DT>{}, std::false_type{});
    }

    // ---- quantize: wavefront w takes tokens w, w + NWT, ...; a lane owns the 16-byte pieces lane, lane + 64, ...
    const int nchunk = K >> 3;
    for (int m = TENSOR ? M : wave; m < M; m += NWT) {
        const uint4* row = reinterpret_cast<const uint4*>(a.x + (int64_t)m * a.ldx);
        uint4 cache[kRowChunks];
        float amax = 0.f;
#pragma unroll
        for (int c = 0; c < kRowChunks; c++) {
            const int i = lane + c * kWave;
            cache[c] = i < nchunk ? row[i] : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int c = 0; c < kRowChunks; c++) amax = max_nonneg(amax, absmax8(cache[c], DT == LLMQ_BF16));
        for (int i = lane + kRowChunks * kWave; i < nchunk; i += kWave) amax = max_nonneg(amax, absmax8(row[i], DT == LLMQ_BF16));
        amax = wave_max(amax);
        const float s = scale_from_amax<DT, MODE>(amax), inv_s = 1.0f / s;
        if (lane == 0) {
            s_scale[m] = s;
            if (a.scale_dump && blockIdx.x == 0) a.scale_dump[m] = s;
        }
        uint2* qrow = reinterpret_cast<uint2*>(smem + m * row_bytes);
        uint2* qdump = (a.q_dump && blockIdx.x == 0) ? reinterpret_cast<uint2*>(a.q_dump + (int64_t)m * K) : nullptr;
        auto codes = [&](auto fin_c) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < kRowChunks; c++) {
                const int i = lane + c * kWave;
                if (i < nchunk) {
                    const uint2 q = quant8<DT, MODE, Q_DT, decltype(fin_c)::value>(cache[c], s, inv_s);
                    qrow[i] = q;
                    if (qdump) qdump[i] = q;
                }
            }
            for (int i = lane + kRowChunks * kWave; i < nchunk; i += kWave) {
                const uint2 q = quant8<DT, MODE, Q_DT, decltype(fin_c)::value>(row[i], s, inv_s);
                qrow[i] = q;
                if (qdump) qdump[i] = q;
            }
        };
        if (amax < __builtin_inff() && s > 0.f) codes(std::true_type{});  // wavefront-uniform: no quotient can be NaN
        else codes(std::false_type{});
    }
    __syncthreads();
    const uint8_t* arow = smem + min(r16, M - 1) * row_bytes + kq * LB;  // rows past M repeat the last token; never stored

    acc_t acc[T];
#pragma unroll
    for (int t = 0; t < T; t++) acc[t] = acc_t{0, 0, 0, 0};

    auto compute_batch = [&](int s0, const Batch& d) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < D; i++) {
            const bool live = s0 + i < s_end;  // wavefront-uniform: steps past the run contribute nothing
            u4 bm[T][P], am[P];
#pragma unroll
            for (int p = 0; p < P; p++) {
                const int koff = (s0 + i) * KSTEP + kq * LB + 16 * p;
                const bool ok = live && koff < K;
                const uint32_t keep = ok ? 0xffffffffu : 0u;
#pragma unroll
                for (int t = 0; t < T; t++) bm[t][p] = d.b[i][t][p] & keep;
                am[p] = *reinterpret_cast<const u4*>(arow + (ok ? (s0 + i) * KSTEP + 16 * p : -(kq * LB)));
            }
#pragma unroll
            for (int t = 0; t < T; t++) {
                if constexpr (FP8) {
                    const v8i bw = {(int)bm[t][0][0], (int)bm[t][0][1], (int)bm[t][0][2], (int)bm[t][0][3],
                                    (int)bm[t][1][0], (int)bm[t][1][1], (int)bm[t][1][2], (int)bm[t][1][3]};
                    const v8i aw = {(int)am[0][0], (int)am[0][1], (int)am[0][2], (int)am[0][3],
                                    (int)am[1][0], (int)am[1][1], (int)am[1][2], (int)am[1][3]};
                    acc[t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bw, aw, acc[t], 0, 0, 0, 0, 0, 0);
                } else {
                    const v4i bw = {(int)bm[t][0][0], (int)bm[t][0][1], (int)bm[t][0][2], (int)bm[t][0][3]};
                    const v4i aw = {(int)am[0][0], (int)am[0][1], (int)am[0][2], (int)am[0][3]};
                    acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bw, aw, acc[t], 0, 0, 0);
                }
            }
        }
    };

    if (s_begin < s_end) {
#pragma unroll 1
        for (int s = s_begin; s < s_end; s += 2 * D) {
            load_batch(s + D, bb);
            compute_batch(s, ba);
            load_batch(s + 2 * D, ba);
            compute_batch(s + D, bb);
        }
    }

    // ---- the block's wavefronts add up in wavefront order (int32: exact; fp32: fixed order)
    __syncthreads();  // every wavefront is done reading the codes: their memory is reused
    acc_t (*red)[T][kWave] = reinterpret_cast<acc_t (*)[T][kWave]>(smem);
    if (ng < NG) {
#pragma unroll
        for (int t = 0; t < T; t++) red[wave][t][lane] = acc[t];
    }
    __syncthreads();
    for (int idx = tid; idx < NG * T * kWave; idx += NT) {
        const int g = idx / (T * kWave), t = (idx / kWave) % T, l = idx % kWave;
        acc_t sum = red[g * NW][t][l];
#pragma unroll
        for (int w = 1; w < NW; w++) sum += red[g * NW + w][t][l];
        // lane l of that accumulator: token l % 16, four channels from 16 t + 4 (l / 16) of the set
        const int m = l & 15, n = (blockIdx.x * NG + g) * (16 * T) + 16 * t + 4 * (l >> 4);
        if (m >= M || n >= N) continue;
        const float sa = TENSOR ? 1.f : s_scale[m], alpha = TENSOR ? s_scale[0] : 1.f;
        uint16_t h[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int ne = min(n + e, N - 1);
            const float sw = !TENSOR && a.w_scale ? a.w_scale[ne] : 1.f;
            const float bb2 = a.bias ? load_as_f32(a.bias, a.bias_dtype, ne) : 0.f;
            const float v = epi_value((float)sum[e], sa, sw, alpha, bb2);
            h[e] = a.out_dtype == LLMQ_BF16 ? Lo<LLMQ_BF16>::from_f32(v) : Lo<LLMQ_F16>::from_f32(v);
        }
        uint16_t* orow = reinterpret_cast<uint16_t*>(a.out) + (int64_t)m * a.ldo + n;
        if (SRC == SRC_STATIC && a.out_scale) {
            float* frow = reinterpret_cast<float*>(a.out) + (int64_t)m * a.ldo + n;
            const float os = *a.out_scale;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float f = a.out_dtype == LLMQ_BF16 ? Lo<LLMQ_BF16>::to_f32(h[e]) : Lo<LLMQ_F16>::to_f32(h[e]);
                if (n + e < N) frow[e] = fp8_round_trip(f, os);
            }
        } else if (n + 3 < N && ((reinterpret_cast<uintptr_t>(orow) & 7u) == 0)) {
            *reinterpret_cast<uint2*>(orow) = make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < N) orow[e] = h[e];
        }
        if (a.acc_dump) {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < N) {
                    const auto sv = sum[e];  // scalar copy first: a bit cast applied to the vector element itself reads element 0
                    reinterpret_cast<uint32_t*>(a.acc_dump)[(int64_t)m * N + n + e] = __builtin_bit_cast(uint32_t, sv);
                }
        }
    }
}

thread_local int g_force_fused_variant = -1;  // tuning hook (per host thread): 0 = 2 channel tiles x 4 wavefronts, 1 = 1 x 8

template <bool FP8, int DT, int T, int NW, int NG, int NI, int SRC, int CH>
int launch_variant(const FusedArgs& a, hipStream_t st) {
    constexpr int D = FP8 ? 2 : 4;  // steps per batch: ~64 registers per batch
    auto kernel = linear_fused_kernel<FP8, DT, T, NW, NG, NI, D, SRC, CH>;
    const size_t lds = std::max<size_t>((size_t)a.M * (a.K + kRowPad), (size_t)NW * NG * T * kWave * 16);  // codes, then the reduction
    if (lds > 64 * 1024) {
        // per device: the attribute belongs to the loaded code object of the current device
        static bool raised[64] = {};
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return LLMQ_ERR_LAUNCH;
        if (dev < 0 || dev >= 64 || !raised[dev]) {
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024) != hipSuccess)
                return LLMQ_ERR_LAUNCH;
            if (dev >= 0 && dev < 64) raised[dev] = true;
        }
    }
    hipLaunchKernelGGL(kernel, dim3((a.N + 16 * T * NG - 1) / (16 * T * NG)), dim3((NW * NG + NI) * kWave), lds, st, a);
    return launch_status();
}

constexpr int64_t kFewChannels = 4096;       // 256 blocks of 16 channels
constexpr int64_t kMostCodes = 10 * 8192;    // codes that 1024 threads hold in 40 registers each, and their LDS

template <bool FP8, int DT, int SRC>
int launch_fused(const FusedArgs& a, hipStream_t st) {
    const int64_t codes = (int64_t)a.M * a.K;
    if constexpr (SRC == SRC_TOKEN) {
        if (g_force_fused_variant == 0) return launch_variant<FP8, DT, 2, 4, 1, 0, SRC, 1>(a, st);
        if (g_force_fused_variant == 1) return launch_variant<FP8, DT, 1, 8, 1, 0, SRC, 1>(a, st);
        // few channels: a wavefront per row (us, 8 / 16 wavefronts: 8 x 1152 x 896 6.2 / 5.4, 11 x 3072 x 4352 12.3 / 11.0); many: four wavefronts and
        // one channel tile each (two tiles / one: 2 x 9216 x 1792 10.6 / 9.2, 3 x 11392 x 1376 7.8 / 7.0), or two where the blocks of a CU would
        // repeat the quantizer six times and more (3 x 23560 x 1920 11.9 / 13.3, 4 x 26112 x 6784 50.4 / 51.8)
        if (a.N <= kFewChannels) return launch_variant<FP8, DT, 1, 4, 1, 12, SRC, 1>(a, st);
        if (a.N > 16384) return launch_variant<FP8, DT, 2, 4, 1, 0, SRC, 1>(a, st);
        if (a.M <= 4) return launch_variant<FP8, DT, 1, 4, 1, 0, SRC, 1>(a, st);
        return launch_variant<FP8, DT, 1, 4, 2, 0, SRC, 1>(a, st);
    } else {
        if (a.N <= kFewChannels || codes > 32768) {
            if (codes <= 16384) return launch_variant<FP8, DT, 1, 4, 1, 12, SRC, 2>(a, st);
            if (codes <= 32768) return launch_variant<FP8, DT, 1, 4, 1, 12, SRC, 4>(a, st);
            return launch_variant<FP8, DT, 1, 4, 1, 12, SRC, 10>(a, st);
        }
        if (codes <= 8192) return launch_variant<FP8, DT, 1, 4, 1, 0, SRC, 4>(a, st);
        if (codes <= 16384) return launch_variant<FP8, DT, 1, 4, 2, 0, SRC, 4>(a, st);
        return launch_variant<FP8, DT, 1, 4, 2, 0, SRC, 8>(a, st);
    }
}

int64_t tensor_max_tokens(int64_t K) { return K <= 0 ? 0 : std::min<int64_t>(16, 16384 / K); }

// what every entry point refuses
int check_args(const void* x, int x_dtype, int64_t ldx, const uint8_t* B, int64_t ldb, const void* bias, int bias_dtype, const void* out,
               int out_dtype, int64_t ldo, int64_t N, int64_t K) {
    if (!x || !B || !out) return LLMQ_ERR_NULL;
    if (x_dtype != LLMQ_BF16 && x_dtype != LLMQ_F16) return LLMQ_ERR_DTYPE;
    if (out_dtype != LLMQ_BF16 && out_dtype != LLMQ_F16) return LLMQ_ERR_DTYPE;
    if (bias && bias_dtype != LLMQ_BF16 && bias_dtype != LLMQ_F16 && bias_dtype != LLMQ_F32) return LLMQ_ERR_DTYPE;
    if (K == 0 || (K & 15) || (ldx & 7) || (ldb & 15) || ldx < K || ldb < K || ldo < N) return LLMQ_ERR_SHAPE;
    if (N > 0x7fffffffLL || K > 0x7fffffffLL || ldx >= (1 << 22) || ldb >= (1 << 22)) return LLMQ_ERR_SHAPE;
    if (!aligned16(x) || !aligned16(B)) return LLMQ_ERR_ALIGN;
    return LLMQ_OK;
}

template <int SRC>
int dispatch(bool fp8, int x_dtype, const FusedArgs& a, hipStream_t st) {
    if constexpr (SRC != SRC_STATIC) {
        if (!fp8) return x_dtype == LLMQ_BF16 ? launch_fused<false, LLMQ_BF16, SRC>(a, st) : launch_fused<false, LLMQ_F16, SRC>(a, st);
    }
    return x_dtype == LLMQ_BF16 ? launch_fused<true, LLMQ_BF16, SRC>(a, st) : launch_fused<true, LLMQ_F16, SRC>(a, st);
}

int fused_entry(bool fp8, const void* x, int x_dtype, int64_t ldx, const uint8_t* B, int64_t ldb, const float* w_scale,
                const void* bias, int bias_dtype, void* out, int out_dtype, int64_t ldo, int64_t M, int64_t N, int64_t K,
                uint8_t* q_dump, float* scale_dump, void* acc_dump, hipStream_t st, bool tensor = false) {
    if (M < 0 || N < 0 || K < 0) return LLMQ_ERR_SHAPE;
    if (M > 16 || M * (K + kRowPad) > kMaxLdsBytes) return LLMQ_ERR_SHAPE;  // llmq_linear_dynamic_max_tokens(K)
    if (tensor && M > tensor_max_tokens(K)) return LLMQ_ERR_SHAPE;
    if (M == 0 || N == 0) return LLMQ_OK;
    if (tensor && !w_scale) return LLMQ_ERR_NULL;
    const int bad = check_args(x, x_dtype, ldx, B, ldb, bias, bias_dtype, out, out_dtype, ldo, N, K);
    if (bad != LLMQ_OK) return bad;
    if (q_dump && !aligned16(q_dump)) return LLMQ_ERR_ALIGN;
    const FusedArgs a{(const uint16_t*)x, B, w_scale, bias, out, q_dump, scale_dump, acc_dump, ldx, ldb, ldo,
                      (int)M, (int)N, (int)K, bias_dtype, out_dtype, nullptr, nullptr};
    return tensor ? dispatch<SRC_TENSOR>(fp8, x_dtype, a, st) : dispatch<SRC_TOKEN>(fp8, x_dtype, a, st);
}

bool one_launch_fits(int kind, int64_t M, int64_t N, int64_t K) {
    return M >= 1 && M <= 16 && N >= 1 && K >= 16 && K % 16 == 0 && kind >= LLMQ_LINEAR_I8_TOKEN && kind <= LLMQ_LINEAR_FP8_STATIC && M * K <= kMostCodes;
}

}  // namespace
}  // namespace llmq

using namespace llmq;

extern "C" int llmq_linear_dynamic_max_tokens(int64_t K) {
    if (K <= 0) return 0;
    const int64_t fit = kMaxLdsBytes / (K + kRowPad);
    return (int)(fit < 16 ? fit : 16);
}

extern "C" int llmq_linear_dynamic_force_variant(int v) {
    if (v < -1 || v > 1) return LLMQ_ERR_SHAPE;
    g_force_fused_variant = v;
    return LLMQ_OK;
}

extern "C" int llmq_linear_i8_dynamic(const void* x, int x_dtype, int64_t ldx, const int8_t* B, int64_t ldb,
                                      const float* w_scale, const void* bias, int bias_dtype, void* out, int out_dtype,
                                      int64_t ldo, int64_t M, int64_t N, int64_t K, int8_t* q_dump, float* scale_dump,
                                      int32_t* acc_dump, llmq_stream_t stream) {
    return fused_entry(false, x, x_dtype, ldx, (const uint8_t*)B, ldb, w_scale, bias, bias_dtype, out, out_dtype, ldo, M, N, K,
                       (uint8_t*)q_dump, scale_dump, acc_dump, (hipStream_t)stream);
}

extern "C" int llmq_linear_fp8_dynamic(const void* x, int x_dtype, int64_t ldx, const uint8_t* B, int64_t ldb,
                                       const float* w_scale, const void* bias, int bias_dtype, void* out, int out_dtype,
                                       int64_t ldo, int64_t M, int64_t N, int64_t K, uint8_t* q_dump, float* scale_dump,
                                       float* acc_dump, llmq_stream_t stream) {
    return fused_entry(true, x, x_dtype, ldx, B, ldb, w_scale, bias, bias_dtype, out, out_dtype, ldo, M, N, K, q_dump,
                       scale_dump, acc_dump, (hipStream_t)stream);
}

// One launch or two.  Measured on an MI355X against quantizer + GEMM, in graphs, weights out of HBM, 4000 random problems of up to 16 tokens.
//
// On the GPU alone (llmq_linear_one_launch_ahead; us, two launches / one): one is ahead as long as the codes that every block makes are few for the
// launch they save.  Per token, a wavefront per row: a short K (0.81 of the time up to 1888 elements), longer rows only with up to 24576 codes (8.1 /
// 7.7 at 2 x 3584 x 3584, 8.1 / 10.0 at 15 x 3584 x 3584, 10.2 / 12.4 at 5 x 688 x 7936).  Per tensor up to 32768 codes (0.79 up to 18416, 0.95 up to 33000, 1.09-1.2 past
// that: 8.3 / 11.6 at 14 x 416 x 4096, 9.0 / 12.3 at 16 x 896 x 4864), with a static scale up to 20480.  With more than 4096 channels each CU repeats
// the quantizer and the GEMM alone streams at 5-6 TB/s, so few codes and short rows (8.9 / 7.4 at 7 x 9728 x 896; 19.4 / 23.4 at 2 x 8704 x 6464, 38.7 / 46.1
// at 1 x 14200 x 13088), and past 16384 channels only where the GEMM has a ragged K (9.1 / 8.0 at 2 x 22368 x 400, 13.3 / 11.6 at 3 x 18064 x 1600; 12.2 / 18.2 at
// 1 x 26176 x 1280).
//
// From a program's own loop (llmq_linear_one_launch_preferred) a second launch takes the host 4 us more, 10 instead of 6, and a decoder layer of small
// projections waits for the host: one launch also where it costs the GPU less than that, up to 49152 codes and with up to 1024 channels all (a layer
// of hidden size 896, 10 tokens: 34.5, with two launches for gate_up and down 42.3), but not for rows so long that the GPU takes more than 10 us either
// way (14.1 / 16.0 at 2 x 312 x 17408, 15.0 / 17.5 at 2 x 1040 x 19456).  The larger of GPU and host time of the same problems is 1.0 % over that of the better choice.
extern "C" int llmq_linear_one_launch_preferred(int kind, int64_t M, int64_t N, int64_t K) {
    if (!one_launch_fits(kind, M, N, K)) return 0;
    const int64_t codes = M * K;
    if (kind == LLMQ_LINEAR_I8_TOKEN || kind == LLMQ_LINEAR_FP8_TOKEN) {
        if (K >= 8192) return 0;
        if (N <= kFewChannels) return M <= 4 || (codes <= 49152 && K <= 6144);
        if (N > 16384) return M >= 2 && M <= 4 && N <= 24576 && K % 128 != 0 && codes <= 4800;
        return M <= 4 && codes <= (N <= 8192 ? 14336 : 8192);
    }
    if (kind == LLMQ_LINEAR_FP8_STATIC) return N <= kFewChannels ? codes <= 32768 : codes <= 14336 && K < 8192 && N <= 16384;
    if (N > kFewChannels) return codes <= 8192 || (K < 6144 && codes <= (N <= 8192 ? 28672 : 16384) && N <= 16384);
    return K <= 5120 ? codes <= 49152 || N <= 1024 : codes <= 32768;
}

extern "C" int llmq_linear_one_launch_ahead(int kind, int64_t M, int64_t N, int64_t K) {
    if (!llmq_linear_one_launch_preferred(kind, M, N, K)) return 0;
    const int64_t codes = M * K;
    if (kind == LLMQ_LINEAR_I8_TOKEN || kind == LLMQ_LINEAR_FP8_TOKEN) return K <= 1888 || (N <= kFewChannels && K <= 5824 && codes <= 24576);
    if (kind == LLMQ_LINEAR_FP8_STATIC) return codes <= (N <= kFewChannels ? 20480 : 9216);
    return codes <= 32768 && N <= 16384;
}

extern "C" int llmq_linear_one_launch(int kind, const void* x, int x_dtype, int64_t ldx, const void* B, int64_t ldb, const float* w_scale,
                                      const float* in_scale, const void* bias, int bias_dtype, const float* out_scale, void* out, int out_dtype,
                                      int64_t ldo, int64_t M, int64_t N, int64_t K, llmq_stream_t stream) {
    if (M < 0 || N < 0 || K < 0 || kind < LLMQ_LINEAR_I8_TOKEN || kind > LLMQ_LINEAR_FP8_STATIC) return LLMQ_ERR_SHAPE;
    if (M == 0 || N == 0) return LLMQ_OK;
    if (!one_launch_fits(kind, M, N, K)) return LLMQ_ERR_SHAPE;
    const bool is_static = kind == LLMQ_LINEAR_FP8_STATIC, token = kind == LLMQ_LINEAR_I8_TOKEN || kind == LLMQ_LINEAR_FP8_TOKEN;
    if ((!token && !w_scale) || (is_static && !in_scale)) return LLMQ_ERR_NULL;
    if (out_scale && !is_static) return LLMQ_ERR_DTYPE;
    const int bad = check_args(x, x_dtype, ldx, (const uint8_t*)B, ldb, bias, bias_dtype, out, out_dtype, ldo, N, K);
    if (bad != LLMQ_OK) return bad;
    const FusedArgs a{(const uint16_t*)x, (const uint8_t*)B, w_scale, bias, out, nullptr, nullptr, nullptr, ldx, ldb, ldo,
                      (int)M, (int)N, (int)K, bias_dtype, out_dtype, in_scale, out_scale};
    const bool fp8 = kind == LLMQ_LINEAR_FP8_TOKEN || kind == LLMQ_LINEAR_FP8_TENSOR || is_static;
    hipStream_t st = (hipStream_t)stream;
    return is_static ? dispatch<SRC_STATIC>(fp8, x_dtype, a, st) : token ? dispatch<SRC_TOKEN>(fp8, x_dtype, a, st) : dispatch<SRC_TENSOR>(fp8, x_dtype, a, st);
}

extern "C" int llmq_linear_per_tensor_max_tokens(int64_t K) { return (int)tensor_max_tokens(K); }

extern "C" int llmq_linear_per_tensor_dynamic(int fp8, const void* x, int x_dtype, int64_t ldx, const void* B, int64_t ldb,
                                              const float* w_scale, const void* bias, int bias_dtype, void* out, int out_dtype,
                                              int64_t ldo, int64_t M, int64_t N, int64_t K, llmq_stream_t stream) {
    return fused_entry(fp8 != 0, x, x_dtype, ldx, (const uint8_t*)B, ldb, w_scale, bias, bias_dtype, out, out_dtype, ldo, M, N, K,
                       nullptr, nullptr, nullptr, (hipStream_t)stream, true);
}
