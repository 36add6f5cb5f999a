// Activation quantizers (int8 SmoothQuant and OCP e4m3fn FP8), one fused HIP kernel each.
//
// The reference runs these as chains of eager torch ops in the activation dtype
// (nn_models/modules/linear/linear_sq.py:44-65, nn_models/modules/linear/linear_fp8.py:11-63):
//   scale = round_dt( max(absmax, round_dt(floor)) / qmax )
//   q     = narrow( clamp( round_dt( x / scale ) ) )
// The kernels reproduce exactly that sequence of roundings.  They are HBM-bound:
// 2 bytes read + 1 byte written per element, one block (of 128 to 1024 threads, row_shape below) or wavefront per row, the row
// held in registers between the absmax pass and the quantize pass so x is read from HBM once.
#include <type_traits>

#include "llmq_common.h"
#include "quant_math.h"

namespace llmq {
namespace {

constexpr int kThreads = 256;
constexpr int kNW = kThreads / kWave;
constexpr int kMaxPartials = 1024;  // per-tensor absmax partials (one per stage-1 block)

enum { SCALE_ROW = 0, SCALE_TENSOR = 1, SCALE_STATIC = 2 };

// The factor the GEMM behind a per-tensor quantizer applies: activation scale x weight scale, formed by the quantizer
// (one thread) instead of by separate elementwise launches.  round_dt: the product is rounded to the activation dtype
// (SmoothQuant, linear_sq.py:127); otherwise it stays fp32 (linear_fp8.py:199-221, 296-308).  out may be null.
struct TensorAlpha {
    const float* w_scale;
    float* out;
    int round_dt;
};
template <int DT>
__device__ __forceinline__ void store_alpha(const TensorAlpha& ta, float s) {
    if (!ta.out) return;
    const float a = s * ta.w_scale[0];
    ta.out[0] = ta.round_dt ? Lo<DT>::round(a) : a;
}

// One block of NT threads per row.  NC > 0: the row's 16-byte chunks (8 elements) are kept in NC
// registers per thread between the two passes; NC == 0: rows of any length, second pass
// re-reads x (served by L2).  A tensor-wide or static scale needs no second look at the row: with up to 512 rows it is held in registers
// all the same, requested ahead of the scale; with more NC == 0, whose fewer registers keep more rows in flight (launch_rows).
template <int DT, int MODE, int SCALE, int NC, int NT = kThreads>
__global__ __launch_bounds__(NT) void quant_rows_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, int64_t K, uint8_t* __restrict__ q,
    void* __restrict__ scale_out, int scale_dtype, const float* __restrict__ aux, int n_aux,
    int static_f32, float floor, TensorAlpha ta) {
    __shared__ float smem[NT / kWave];
    const int64_t row = blockIdx.x;
    const int tid = threadIdx.x;
    const int nchunk = (int)(K >> 3);
    const uint4* xr = reinterpret_cast<const uint4*>(x + row * ldx);
    uint2* qr = reinterpret_cast<uint2*>(q + row * K);

    uint4 cache[NC > 0 ? NC : 1];
    float s;
    bool fin = false;  // block-uniform: the absmax behind the scale is finite, so no quotient can be NaN
    // The row is requested before the scale is known, also where it comes from elsewhere: its latency runs beside that of the partials
    // or of the scale.
    if (NC > 0) {
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int i = tid + c * NT;
            cache[c] = (i < nchunk) ? xr[i] : make_uint4(0, 0, 0, 0);
        }
    }
    if (SCALE == SCALE_ROW) {
        float amax = 0.f;
        if (NC > 0) {
#pragma unroll
            for (int c = 0; c < NC; c++) amax = max_nonneg(amax, absmax8(cache[c], DT == LLMQ_BF16));
        } else {
            for (int i = tid; i < nchunk; i += NT) amax = max_nonneg(amax, absmax8(xr[i], DT == LLMQ_BF16));
        }
        amax = block_max<NT / kWave>(amax, smem);
        s = scale_from_amax<DT, MODE>(amax, floor);
        fin = amax < __builtin_inff() && s > 0.f;  // (the fp8 floor rounds to 0 in fp16: an all-zero row has scale 0 and 0 / 0)
    } else if (SCALE == SCALE_TENSOR) {
        float amax = 0.f;
        for (int i = tid; i < n_aux; i += NT) amax = max_nonneg(amax, aux[i]);
        amax = block_max<NT / kWave>(amax, smem);
        s = scale_from_amax<DT, MODE>(amax, floor);
        fin = amax < __builtin_inff() && s > 0.f;  // (the fp8 floor rounds to 0 in fp16: an all-zero row has scale 0 and 0 / 0)
    } else {
        s = aux[0];
    }
    if (SCALE != SCALE_STATIC && tid == 0 && (SCALE == SCALE_ROW || row == 0)) {
        const int64_t o = SCALE == SCALE_ROW ? row : 0;
        if (scale_dtype == LLMQ_F32) ((float*)scale_out)[o] = s;
        else ((uint16_t*)scale_out)[o] = Lo<DT>::from_f32(s);
    }
    if (SCALE != SCALE_ROW && row == 0 && tid == 0) store_alpha<DT>(ta, s);
    const float inv_s = 1.0f / s;
    auto store_row = [&](auto quot_c, auto fin_c) __attribute__((always_inline)) {
        constexpr int QUOT = decltype(quot_c)::value;
        constexpr bool FIN = decltype(fin_c)::value;
        if (NC > 0) {
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const int i = tid + c * NT;
                if (i < nchunk) qr[i] = quant8<DT, MODE, QUOT, FIN>(cache[c], s, inv_s);
            }
        } else {
            for (int i = tid; i < nchunk; i += NT) qr[i] = quant8<DT, MODE, QUOT, FIN>(xr[i], s, inv_s);
        }
    };
    if (SCALE == SCALE_STATIC) {
        if (static_f32 && near_scale(s)) store_row(std::integral_constant<int, Q_NEAR_F32>{}, std::false_type{});
        else if (static_f32) store_row(std::integral_constant<int, Q_DIV_F32>{}, std::false_type{});
        else store_row(std::integral_constant<int, Q_DIV_DT>{}, std::false_type{});
    } else if (fin) {
        store_row(std::integral_constant<int, Q_DT>{}, std::true_type{});
    } else {
        store_row(std::integral_constant<int, Q_DT>{}, std::false_type{});
    }
}

// One wavefront per row, for rows of at most 64 * NCW chunks: no block barrier, the reductions are wavefront
// butterflies, and the four rows of a block are independent, so four times as many rows are in flight per CU.
template <int DT, int MODE, int NCW>
__global__ __launch_bounds__(kThreads) void quant_rows_wave_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, int64_t K, int64_t M, uint8_t* __restrict__ q,
    void* __restrict__ scale_out, int scale_dtype, float floor) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t row = (int64_t)blockIdx.x * kNW + threadIdx.x / kWave;
    if (row >= M) return;  // wavefront-uniform; the kernel has no barrier
    const int nchunk = (int)(K >> 3);
    const uint4* xr = reinterpret_cast<const uint4*>(x + row * ldx);
    uint2* qr = reinterpret_cast<uint2*>(q + row * K);
    uint4 cache[NCW];
#pragma unroll
    for (int c = 0; c < NCW; c++) {
        const int i = lane + c * kWave;
        cache[c] = (i < nchunk) ? xr[i] : make_uint4(0, 0, 0, 0);
    }
    float amax = 0.f;
#pragma unroll
    for (int c = 0; c < NCW; c++) amax = max_nonneg(amax, absmax8(cache[c], DT == LLMQ_BF16));
    amax = wave_max(amax);
    const float s = scale_from_amax<DT, MODE>(amax, floor);
    if (lane == 0) {
        if (scale_dtype == LLMQ_F32) ((float*)scale_out)[row] = s;
        else ((uint16_t*)scale_out)[row] = Lo<DT>::from_f32(s);
    }
    const float inv_s = 1.0f / s;
    if (amax < __builtin_inff() && s > 0.f) {  // wavefront-uniform: no quotient can be NaN
#pragma unroll
        for (int c = 0; c < NCW; c++) {
            const int i = lane + c * kWave;
            if (i < nchunk) qr[i] = quant8<DT, MODE, Q_DT, true>(cache[c], s, inv_s);
        }
    } else {
#pragma unroll
        for (int c = 0; c < NCW; c++) {
            const int i = lane + c * kWave;
            if (i < nchunk) qr[i] = quant8<DT, MODE, Q_DT>(cache[c], s, inv_s);
        }
    }
}

// Stage 1 of the per-tensor quantizers: absmax partials, one per block.  The tensor's chunks, row after row, are cut into
// units of kUnit; a thread takes kUnitLoads independent 16-byte loads of a unit.  HBM-bound: 8192 x 3584 12.9 us (4.6 TB/s;
// one load at a time with a division per chunk 14.2), 4096 x 18944 34.1 us (36.4).
// STRIDED: rows of cpr chunks lie ldx apart.  A thread divides once per unit to find its first chunk and steps from there:
// step_rows, step_chunks = kThreads / cpr, kThreads % cpr.  Units follow the chunks and not the rows, so that short rows fill
// them too.
constexpr int kUnitLoads = 8, kUnit = kUnitLoads * kThreads;
template <int DT, bool STRIDED>
__global__ __launch_bounds__(kThreads) void absmax_partials_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, int64_t cpr, int64_t total, int64_t step_rows, int64_t step_chunks,
    float* __restrict__ partials) {
    __shared__ float smem[kNW];
    const uint4* first = reinterpret_cast<const uint4*>(x);
    const uint4* last = STRIDED ? reinterpret_cast<const uint4*>(x + (total / cpr - 1) * ldx) + (cpr - 1) : first + (total - 1);
    float amax = 0.f;
    for (int64_t base = (int64_t)blockIdx.x * kUnit; base < total; base += (int64_t)gridDim.x * kUnit) {
        const int64_t at = base + threadIdx.x;
        int64_t r = 0, c = at;
        if (STRIDED) {
            r = total <= 0xffffffffLL ? (int64_t)((uint32_t)at / (uint32_t)cpr) : at / cpr;
            c = at - r * cpr;
        }
        uint4 v[kUnitLoads];
#pragma unroll
        for (int i = 0; i < kUnitLoads; i++) {
            const uint4* src = STRIDED ? reinterpret_cast<const uint4*>(x + r * ldx) + c : first + (at + i * kThreads);
            v[i] = *(at + i * kThreads < total ? src : last);  // past the end: the last chunk again, which changes no maximum
            if (STRIDED) {
                r += step_rows;
                c += step_chunks;
                if (c >= cpr) c -= cpr, r++;
            }
        }
#pragma unroll
        for (int i = 0; i < kUnitLoads; i++) amax = max_nonneg(amax, absmax8(v[i], DT == LLMQ_BF16));
    }
    amax = block_max<kNW>(amax, smem);
    if (threadIdx.x == 0) partials[blockIdx.x] = amax;
}

// Per-tensor quantizer of a small contiguous tensor in one launch: every block reduces the whole tensor by itself (it
// sits in L2; what is saved is a launch and the gap in front of it), then quantizes its own 1024 chunks.  Bound by the
// latency of launch, loads and reduction.
constexpr int kSmallThreads = 1024;
template <int DT, int MODE>
__global__ __launch_bounds__(kSmallThreads) void quant_tensor_small_kernel(
    const uint4* __restrict__ x, int total, uint2* __restrict__ q, void* __restrict__ scale_out, int scale_dtype,
    float floor, TensorAlpha ta) {
    __shared__ float smem[kSmallThreads / kWave];
    const int tid = threadIdx.x, mine = blockIdx.x * kSmallThreads + tid;
    const uint4 own = x[mine < total ? mine : total - 1];
    float amax = 0.f;
    for (int i0 = tid; i0 < total; i0 += kUnitLoads * kSmallThreads) {
        uint4 v[kUnitLoads];
#pragma unroll
        for (int i = 0; i < kUnitLoads; i++) {
            const int c = i0 + i * kSmallThreads;
            v[i] = x[c < total ? c : total - 1];
        }
#pragma unroll
        for (int i = 0; i < kUnitLoads; i++) amax = max_nonneg(amax, absmax8(v[i], DT == LLMQ_BF16));
    }
    amax = block_max<kSmallThreads / kWave>(amax, smem);
    const float s = scale_from_amax<DT, MODE>(amax, floor);
    if (mine == 0) {
        if (scale_dtype == LLMQ_F32) ((float*)scale_out)[0] = s;
        else ((uint16_t*)scale_out)[0] = Lo<DT>::from_f32(s);
        store_alpha<DT>(ta, s);
    }
    if (mine >= total) return;
    if (amax < __builtin_inff() && s > 0.f) q[mine] = quant8<DT, MODE, Q_DT, true>(own, s, 1.0f / s);
    else q[mine] = quant8<DT, MODE, Q_DT>(own, s, 1.0f / s);
}

// ---- RMSNorm fused with the per-token quantizer --------------------------------------------
// The reference normalises (nn_models/modules/nonlinear/norm.py:10-16) and then quantizes the result in
// the first Linear of the block (nn_models/modules/nonlinear/block.py:68,76 -> linear_sq.py:55-65 /
// linear_fp8.py:40-63): two round trips of the activations through HBM.  Here a row is read once, kept
// in registers, normalised, (optionally) written back as y, and quantized:
//   h = fp32(x);  inv = 1 / sqrt(mean(h^2) + eps);  n = round_dt(h * inv);  y = round_dt(w * n)
//   then exactly the per-token quantizer above on y.
// Everything after `inv` is bit-identical to the reference evaluated with the same inv; inv itself
// depends on the summation order of mean() and can differ from another order in the last bits.  The order here: LANES running sums, sum t
// an FMA chain over the row's 16-byte chunks t, t + LANES, ..; a butterfly over each 64 of them; the results of the 64s in order.  LANES
// follows from the size alone and not from the block that does the work (norm_shape below).
template <int DT>
__device__ __forceinline__ float sumsq8(uint4 r, float acc) {
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float a = Lo<DT>::to_f32((uint16_t)(w[i] & 0xffffu)), b = Lo<DT>::to_f32((uint16_t)(w[i] >> 16));
        acc = fmaf(a, a, acc);
        acc = fmaf(b, b, acc);
    }
    return acc;
}

template <int DT>
__device__ __forceinline__ uint4 norm8(uint4 r, uint4 wv, float inv) {
    const uint32_t x[4] = {r.x, r.y, r.z, r.w}, w[4] = {wv.x, wv.y, wv.z, wv.w};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        // The reference rounds the product to fp32 and then to the activation dtype.  Keep the fp32 product
        // opaque so that the compiler cannot fuse multiply and narrowing into one mixed-precision
        // instruction, which rounds once and lands on the other side of a tie now and then.  The two narrowings of a
        // pair share one packed conversion.
        float p0 = Lo<DT>::lo_f32(x[i]) * inv;
        float p1 = Lo<DT>::hi_f32(x[i]) * inv;
        asm volatile("" : "+v"(p0), "+v"(p1));
        const uint32_t n = Lo<DT>::pack2(p0, p1);
        // (the product of two 16-bit floats is exact in fp32: narrowing it rounds once however it is compiled)
        o[i] = Lo<DT>::pack2(Lo<DT>::lo_f32(w[i]) * Lo<DT>::lo_f32(n), Lo<DT>::hi_f32(w[i]) * Lo<DT>::hi_f32(n));
    }
    return make_uint4(o[0], o[1], o[2], o[3]);
}

// QMODE: -1 = no quantizer (plain RMSNorm), MODE_I8, MODE_F8.  G = 2: two halves of LANES threads; thread t of the lower one owns the chunks
// t + c LANES, of the upper one t + (NC + c) LANES.  The upper half reads the lower one's chunks as well and forms the running sums alone: a
// wait for the lower half's through LDS takes longer (one-token layer 50.4 / 49.6 us).
template <int DT, int QMODE, int NC, int NT = kThreads, int G = 1>
__global__ __launch_bounds__(NT) void rmsnorm_quant_rows_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, int64_t K, const uint16_t* __restrict__ weight, float eps,
    uint16_t* __restrict__ y, uint8_t* __restrict__ q, void* __restrict__ scale_out, int scale_dtype,
    float* __restrict__ inv_out) {
    constexpr int QM = QMODE < 0 ? MODE_I8 : QMODE, LANES = NT / G;
    static_assert(LANES % kWave == 0 && (G == 1 || (G == 2 && NC > 0)), "halves of whole wavefronts, rows in registers");
    __shared__ float smem[NT / kWave];
    const int64_t row = blockIdx.x;
    const int tid = threadIdx.x, upper = G > 1 ? __builtin_amdgcn_readfirstlane(tid / LANES) : 0;
    const int first = tid + upper * (NC - 1) * LANES;  // the thread's first chunk; the others follow LANES apart
    const int nchunk = (int)(K >> 3);
    const uint4* xr = reinterpret_cast<const uint4*>(x + row * ldx);
    const uint4* wr = reinterpret_cast<const uint4*>(weight);
    uint4* yr = y ? reinterpret_cast<uint4*>(y + row * K) : nullptr;
    uint2* qr = reinterpret_cast<uint2*>(q + row * K);

    uint4 cache[NC > 0 ? NC : 1];
    float ss = 0.f;
    if (NC > 0) {
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int i = first + c * LANES;
            cache[c] = (i < nchunk) ? xr[i] : make_uint4(0, 0, 0, 0);
        }
        if (upper) {
            uint4 low[NC > 0 ? NC : 1];  // (a lower chunk past the row has no upper one behind it)
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const int i = tid + (c - 1) * LANES;
                low[c] = (i < nchunk) ? xr[i] : make_uint4(0, 0, 0, 0);
            }
#pragma unroll
            for (int c = 0; c < NC; c++) ss = sumsq8<DT>(low[c], ss);
        }
#pragma unroll
        for (int c = 0; c < NC; c++) ss = sumsq8<DT>(cache[c], ss);
    } else {
        for (int i = tid; i < nchunk; i += NT) ss = sumsq8<DT>(xr[i], ss);
    }
    // the last LANES threads hold the sums
    ss = block_sum<LANES / kWave>(ss, smem, (G - 1) * (LANES / kWave));
    const float inv = 1.0f / sqrtf(ss / (float)K + eps);
    if (inv_out && tid == 0) inv_out[row] = inv;

    float amax = 0.f;
    if (NC > 0) {
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int i = first + c * LANES;
            if (i < nchunk) {
                cache[c] = norm8<DT>(cache[c], wr[i], inv);
                if (yr) yr[i] = cache[c];
                amax = max_nonneg(amax, absmax8(cache[c], DT == LLMQ_BF16));
            }
        }
    } else {
        for (int i = tid; i < nchunk; i += NT) {
            const uint4 v = norm8<DT>(xr[i], wr[i], inv);
            if (yr) yr[i] = v;
            amax = max_nonneg(amax, absmax8(v, DT == LLMQ_BF16));
        }
    }
    if (QMODE < 0) return;
    amax = block_max<NT / kWave>(amax, smem);
    const float s = scale_from_amax<DT, QM>(amax);
    if (tid == 0) {
        if (scale_dtype == LLMQ_F32) ((float*)scale_out)[row] = s;
        else ((uint16_t*)scale_out)[row] = Lo<DT>::from_f32(s);
    }
    const float inv_s = 1.0f / s;
    if (NC > 0 && amax < __builtin_inff() && s > 0.f) {  // block-uniform: no quotient can be NaN
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int i = first + c * LANES;
            if (i < nchunk) qr[i] = quant8<DT, QM, Q_DT, true>(cache[c], s, inv_s);
        }
    } else if (NC > 0) {
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int i = first + c * LANES;
            if (i < nchunk) qr[i] = quant8<DT, QM, Q_DT>(cache[c], s, inv_s);
        }
    } else {
        for (int i = tid; i < nchunk; i += NT) qr[i] = quant8<DT, QM, Q_DT>(norm8<DT>(xr[i], wr[i], inv), s, inv_s);
    }
}

// The same with one wavefront per row (see quant_rows_wave_kernel); the sum of squares is a per-lane FMA chain and a
// wavefront butterfly.
template <int DT, int QMODE, int NCW>
__global__ __launch_bounds__(kThreads) void rmsnorm_quant_rows_wave_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, int64_t K, int64_t M, const uint16_t* __restrict__ weight, float eps,
    uint16_t* __restrict__ y, uint8_t* __restrict__ q, void* __restrict__ scale_out, int scale_dtype,
    float* __restrict__ inv_out) {
    constexpr int QM = QMODE < 0 ? MODE_I8 : QMODE;
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t row = (int64_t)blockIdx.x * kNW + threadIdx.x / kWave;
    if (row >= M) return;  // wavefront-uniform; the kernel has no barrier
    const int nchunk = (int)(K >> 3);
    const uint4* xr = reinterpret_cast<const uint4*>(x + row * ldx);
    const uint4* wr = reinterpret_cast<const uint4*>(weight);
    uint4* yr = y ? reinterpret_cast<uint4*>(y + row * K) : nullptr;
    uint2* qr = reinterpret_cast<uint2*>(q + row * K);
    uint4 cache[NCW];
#pragma unroll
    for (int c = 0; c < NCW; c++) {
        const int i = lane + c * kWave;
        cache[c] = (i < nchunk) ? xr[i] : make_uint4(0, 0, 0, 0);
    }
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < NCW; c++) ss = sumsq8<DT>(cache[c], ss);
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)K + eps);
    if (inv_out && lane == 0) inv_out[row] = inv;
    float amax = 0.f;
#pragma unroll
    for (int c = 0; c < NCW; c++) {
        const int i = lane + c * kWave;
        if (i < nchunk) {
            cache[c] = norm8<DT>(cache[c], wr[i], inv);
            if (yr) yr[i] = cache[c];
            amax = max_nonneg(amax, absmax8(cache[c], DT == LLMQ_BF16));
        }
    }
    if (QMODE < 0) return;
    amax = wave_max(amax);
    const float s = scale_from_amax<DT, QM>(amax);
    if (lane == 0) {
        if (scale_dtype == LLMQ_F32) ((float*)scale_out)[row] = s;
        else ((uint16_t*)scale_out)[row] = Lo<DT>::from_f32(s);
    }
    const float inv_s = 1.0f / s;
    if (amax < __builtin_inff() && s > 0.f) {  // wavefront-uniform: no quotient can be NaN
#pragma unroll
        for (int c = 0; c < NCW; c++) {
            const int i = lane + c * kWave;
            if (i < nchunk) qr[i] = quant8<DT, QM, Q_DT, true>(cache[c], s, inv_s);
        }
    } else {
#pragma unroll
        for (int c = 0; c < NCW; c++) {
            const int i = lane + c * kWave;
            if (i < nchunk) qr[i] = quant8<DT, QM, Q_DT>(cache[c], s, inv_s);
        }
    }
}

// Measured with the inputs streamed from HBM: at K = 1024 and 8192 rows the wavefront-per-row kernels take 7.1 us
// (quantizer) / 9.7 us (RMSNorm + quantizer) against 9.3 / 13.7 us for a block per row; at K = 3584 a block per row is
// ahead by 5 % (17.2 against 18.0 us) and by 1.3 us at a few rows, so longer rows keep it.
inline bool wave_rows(int64_t M, int64_t K) { return (K >> 3) <= 2 * kWave && M >= 256; }
// A block per row: threads and chunks per thread, by how many rows have to fill the chip.  A few rows are a chain of latencies (load, two
// reductions, codes), which more threads with less each shorten; many rows are arithmetic that every wavefront repeats per row (reductions,
// scale, reciprocal), which fewer threads with more each spread over more elements.  int8 per-token quantizer, us:
//   257-512 chunks (K = 3584)    512 x 1   256 x 2   128 x 4       1025-2560 chunks (K = 18944)   1024 x 3   512 x 5   256 x 10
//   32 rows                      2.68      2.74      2.72          32 rows                        3.75       3.79      3.99
//   256                          3.03      3.09      3.31          128                            4.47       4.49      4.74
//   512                          3.61      3.60      3.94          512                            8.14       8.22      8.51
//   2048                         7.06      6.35      6.68          2048                           21.2       20.6      20.4
enum RowShape { R512x1, R256x1, R256x2, R128x4, R256x4, R1024x3, R512x5, R256x10, RLong };
inline RowShape row_shape(int64_t M, int64_t K) {
    const int64_t chunks = K >> 3;
    if (chunks <= 256) return R256x1;
    if (chunks <= 512) return M < 400 ? R512x1 : M < 6144 ? R256x2 : R128x4;
    if (chunks <= 1024) return R256x4;
    if (chunks <= 2560) return M <= 256 ? R1024x3 : M <= 1024 ? R512x5 : R256x10;
    return RLong;
}

// RMSNorm: LANES, the order of the sum of squares, is fixed by the size (128 for 257-512 chunks and 256 rows or more, else 256), so wider
// blocks read half of their row twice, and the lines lie elsewhere.  RMSNorm + int8 quantizer, rows in cache, us:
//   K = 3584     512 x 1   256 x 2   128 x 4      K = 18944    512 x 5   256 x 10
//   1 row        2.40      2.80                   32 rows      5.32      6.40
//   128          3.40      3.76                   128          5.76      6.80
//   256                    3.84      4.44         256          6.92      7.32
//   512                    4.24      4.84         512          10.5      8.92
//   768                    4.88      4.96         1024         16.3      17.0
//   1024                   5.56      5.16         2048         28.5      28.4
inline RowShape norm_shape(int64_t M, int64_t K) {
    const int64_t chunks = K >> 3;
    if (chunks <= 256) return R256x1;
    if (chunks <= 512) return M < 256 ? R512x1 : M < 768 ? R256x2 : R128x4;
    if (chunks <= 1024) return R256x4;
    if (chunks <= 2560) return M <= 256 ? R512x5 : R256x10;
    return RLong;
}

template <int DT, int QMODE>
int launch_norm(const void* x, int64_t M, int64_t K, int64_t ldx, const void* weight, float eps, void* y, void* q,
                void* scale, int scale_dtype, float* inv_out, hipStream_t st) {
    const dim3 grid((unsigned)M), block(kThreads);
    if (wave_rows(M, K)) {
        const dim3 wgrid((unsigned)((M + kNW - 1) / kNW));
        const int64_t per_lane = ((K >> 3) + kWave - 1) / kWave;
#define LLMQ_LAUNCH_NCW(NCW)                                                                                          \
    hipLaunchKernelGGL((rmsnorm_quant_rows_wave_kernel<DT, QMODE, NCW>), wgrid, block, 0, st, (const uint16_t*)x, ldx, K, \
                       M, (const uint16_t*)weight, eps, (uint16_t*)y, (uint8_t*)q, scale, scale_dtype, inv_out)
        if (per_lane <= 1) LLMQ_LAUNCH_NCW(1);
        else LLMQ_LAUNCH_NCW(2);
#undef LLMQ_LAUNCH_NCW
        return launch_status();
    }
#define LLMQ_LAUNCH_NCT(NC, NT, G)                                                                                          \
    hipLaunchKernelGGL((rmsnorm_quant_rows_kernel<DT, QMODE, NC, NT, G>), grid, dim3(NT), 0, st, (const uint16_t*)x, ldx, K, \
                       (const uint16_t*)weight, eps, (uint16_t*)y, (uint8_t*)q, scale, scale_dtype, inv_out)
    switch (norm_shape(M, K)) {
        case R512x1: LLMQ_LAUNCH_NCT(1, 512, 2); break;
        case R256x1: LLMQ_LAUNCH_NCT(1, 256, 1); break;
        case R256x2: LLMQ_LAUNCH_NCT(2, 256, 2); break;
        case R128x4: LLMQ_LAUNCH_NCT(4, 128, 1); break;
        case R256x4: LLMQ_LAUNCH_NCT(4, 256, 1); break;
        case R512x5: LLMQ_LAUNCH_NCT(5, 512, 2); break;
        case R256x10: LLMQ_LAUNCH_NCT(10, 256, 1); break;
        default: LLMQ_LAUNCH_NCT(0, 256, 1);
    }
#undef LLMQ_LAUNCH_NCT
    return launch_status();
}

template <int QMODE>
int rmsnorm_entry(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const void* weight, float eps,
                  void* y, void* q, void* scale, int scale_dtype, float* inv_out, hipStream_t st) {
    if (x_dtype != LLMQ_BF16 && x_dtype != LLMQ_F16) return LLMQ_ERR_DTYPE;
    if (M < 0 || K < 0 || ldx < K || (K & 7) || (ldx & 7) || M > 0x7fffffffLL) return LLMQ_ERR_SHAPE;
    if (M == 0) return LLMQ_OK;
    if (K == 0) return LLMQ_ERR_SHAPE;
    if (!x || !weight || (QMODE < 0 ? !y : (!q || !scale))) return LLMQ_ERR_NULL;
    if (QMODE >= 0 && scale_dtype != x_dtype && scale_dtype != LLMQ_F32) return LLMQ_ERR_DTYPE;
    if (!aligned16(x) || !aligned16(weight) || (y && !aligned16(y)) || (q && (reinterpret_cast<uintptr_t>(q) & 7u)))
        return LLMQ_ERR_ALIGN;
    if (x_dtype == LLMQ_BF16)
        return launch_norm<LLMQ_BF16, QMODE>(x, M, K, ldx, weight, eps, y, q, scale, scale_dtype, inv_out, st);
    return launch_norm<LLMQ_F16, QMODE>(x, M, K, ldx, weight, eps, y, q, scale, scale_dtype, inv_out, st);
}

int check_common(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const void* q) {
    if (!x || !q) return (M == 0 || K == 0) ? LLMQ_OK : LLMQ_ERR_NULL;
    if (x_dtype != LLMQ_BF16 && x_dtype != LLMQ_F16) return LLMQ_ERR_DTYPE;
    if (M < 0 || K < 0 || ldx < K || (K & 7) || (ldx & 7) || M > 0x7fffffffLL) return LLMQ_ERR_SHAPE;
    if (!aligned16(x) || (reinterpret_cast<uintptr_t>(q) & 7u)) return LLMQ_ERR_ALIGN;
    return LLMQ_OK;
}

template <int DT, int MODE, int SCALE>
int launch_rows(const void* x, int64_t M, int64_t K, int64_t ldx, void* q, void* scale, int scale_dtype,
                const float* aux, int n_aux, int static_f32, float floor, const TensorAlpha& ta, hipStream_t st) {
    const dim3 grid((unsigned)M), block(kThreads);
    const uint16_t* xp = (const uint16_t*)x;
    uint8_t* qp = (uint8_t*)q;
    if (SCALE == SCALE_ROW && wave_rows(M, K)) {
        const dim3 wgrid((unsigned)((M + kNW - 1) / kNW));
        const int64_t per_lane = ((K >> 3) + kWave - 1) / kWave;
#define LLMQ_LAUNCH_NCW(NCW) \
    hipLaunchKernelGGL((quant_rows_wave_kernel<DT, MODE, NCW>), wgrid, block, 0, st, xp, ldx, K, M, qp, scale, scale_dtype, floor)
        if (per_lane <= 1) LLMQ_LAUNCH_NCW(1);
        else LLMQ_LAUNCH_NCW(2);
#undef LLMQ_LAUNCH_NCW
        return launch_status();
    }
#define LLMQ_LAUNCH_NCT(NC, NT) \
    hipLaunchKernelGGL((quant_rows_kernel<DT, MODE, SCALE, NC, NT>), grid, dim3(NT), 0, st, xp, ldx, K, qp, scale, scale_dtype, aux, n_aux, static_f32, floor, ta)
    // A scale that comes from elsewhere: rows in registers hide their latency behind the partials' or the scale's while a block or two per CU
    // cover the rows; with more, blocks that loop and need fewer registers are ahead.  Loop of 256 threads / rows in registers, us,
    // absmax + quantizer (static scale):
    //            K = 3584                    9728                        18944
    //   64 rows  4.82 / 4.77 (2.58 / 2.29)   6.86 / 5.49 (4.03 / 2.96)   8.74 / 6.37 (7.56 / 4.60)
    //   200      5.73 / 5.45 (2.82 / 2.53)   7.23 / 6.13 (5.02 / 3.64)   10.0 / 7.84 (8.12 / 5.61)
    //   512      6.27 / 6.06 (3.66 / 3.71)   9.15 / 8.67 (6.25 / 6.00)   13.8 / 13.4 (12.2 / 10.4)
    //   1000     7.40 / 7.59 (4.65 / 4.80)   12.7 / 13.4 (9.72 / 9.29)   19.7 / 20.3 (16.0 / 16.3)
    switch (SCALE != SCALE_ROW && M > 512 ? RLong : row_shape(M, K)) {
        case R512x1: LLMQ_LAUNCH_NCT(1, 512); break;
        case R256x1: LLMQ_LAUNCH_NCT(1, 256); break;
        case R256x2: LLMQ_LAUNCH_NCT(2, 256); break;
        case R128x4: LLMQ_LAUNCH_NCT((SCALE == SCALE_ROW ? 4 : 0), (SCALE == SCALE_ROW ? 128 : 256)); break;  // (M >= 6144: rows by token only)
        case R256x4: LLMQ_LAUNCH_NCT(4, 256); break;
        case R1024x3: LLMQ_LAUNCH_NCT(3, 1024); break;
        case R512x5: LLMQ_LAUNCH_NCT(5, 512); break;
        case R256x10: LLMQ_LAUNCH_NCT((SCALE == SCALE_ROW ? 10 : 0), 256); break;  // (M > 1024: the same)
        default: LLMQ_LAUNCH_NCT(0, 256);
    }
    return launch_status();
}

template <int MODE, int SCALE>
int dispatch_rows(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, void* q, void* scale,
                  int scale_dtype, const float* aux, int n_aux, int static_f32, float floor, const TensorAlpha& ta,
                  hipStream_t st) {
    if (x_dtype == LLMQ_BF16)
        return launch_rows<LLMQ_BF16, MODE, SCALE>(x, M, K, ldx, q, scale, scale_dtype, aux, n_aux, static_f32, floor, ta, st);
    return launch_rows<LLMQ_F16, MODE, SCALE>(x, M, K, ldx, q, scale, scale_dtype, aux, n_aux, static_f32, floor, ta, st);
}

// Largest contiguous tensor (in chunks of 8 elements) that the one-launch per-tensor quantizer takes.  Measured (K = 3584,
// back to back, one launch / two launches): 16 rows 3.7 / 6.2 us, 32 rows 4.6 / 6.8, 64 rows 6.4 / 6.8, 128 rows 10.5 / 6.9:
// every block's pass over the whole tensor costs more than a launch from about 28000 chunks on.
constexpr int64_t kSmallChunks = 16384;

template <int DT, int MODE>
int per_tensor_dt(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, void* q, void* scale, int scale_dtype,
                  float* partials, float floor, const TensorAlpha& ta, hipStream_t st) {
    const bool contiguous = ldx == K || M == 1;
    const int64_t total = M * (K >> 3);
    if (contiguous && total <= kSmallChunks) {
        hipLaunchKernelGGL((quant_tensor_small_kernel<DT, MODE>), dim3((unsigned)((total + kSmallThreads - 1) / kSmallThreads)),
                           dim3(kSmallThreads), 0, st, (const uint4*)x, (int)total, (uint2*)q, scale, scale_dtype, floor, ta);
        return launch_status();
    }
    const int64_t cpr = K >> 3, units = (total + kUnit - 1) / kUnit;
    const int nblk = (int)(units < kMaxPartials ? units : kMaxPartials);
    if (contiguous)
        hipLaunchKernelGGL((absmax_partials_kernel<DT, false>), dim3(nblk), dim3(kThreads), 0, st, (const uint16_t*)x, ldx, cpr,
                           total, 0, 0, partials);
    else
        hipLaunchKernelGGL((absmax_partials_kernel<DT, true>), dim3(nblk), dim3(kThreads), 0, st, (const uint16_t*)x, ldx, cpr,
                           total, kThreads / cpr, kThreads % cpr, partials);
    if (launch_status() != LLMQ_OK) return LLMQ_ERR_LAUNCH;
    return dispatch_rows<MODE, SCALE_TENSOR>(x, x_dtype, M, K, ldx, q, scale, scale_dtype, partials, nblk, 0, floor, ta, st);
}

template <int MODE>
int per_tensor(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, void* q, void* scale,
               int scale_dtype, void* ws, size_t ws_bytes, float floor, const TensorAlpha& ta, hipStream_t st) {
    if (!ws || ws_bytes < kMaxPartials * sizeof(float)) return LLMQ_ERR_WORKSPACE;
    if (x_dtype == LLMQ_BF16)
        return per_tensor_dt<LLMQ_BF16, MODE>(x, x_dtype, M, K, ldx, q, scale, scale_dtype, (float*)ws, floor, ta, st);
    return per_tensor_dt<LLMQ_F16, MODE>(x, x_dtype, M, K, ldx, q, scale, scale_dtype, (float*)ws, floor, ta, st);
}

// Per-output-channel int8 weight quantizer (an offline step: one pass when a module is built).  One block per
// row of W [N, K]; any K, any 16-bit or fp32 dtype; arithmetic in the dtype of W as the reference's tensor ops do on
// the GPU: scale = round_dt(absmax / 127) with no floor (an all-zero row gives 0 / 0 = NaN, which narrows to 0),
// q = clamp(rint(round_dt(w / scale)), -128, 127), true division.
template <int DT>
__device__ __forceinline__ float wq_load(const void* w, int64_t i) {
    if (DT == LLMQ_F32) return reinterpret_cast<const float*>(w)[i];
    return Lo<DT == LLMQ_F32 ? LLMQ_BF16 : DT>::to_f32(reinterpret_cast<const uint16_t*>(w)[i]);
}
template <int DT>
__device__ __forceinline__ float wq_round(float v) {
    if (DT == LLMQ_F32) return v;
    return Lo<DT == LLMQ_F32 ? LLMQ_BF16 : DT>::round(v);
}
template <int DT>
__global__ __launch_bounds__(kThreads) void quant_weight_rows_kernel(const void* __restrict__ w, int64_t ldw, int64_t K,
                                                                      int8_t* __restrict__ q, void* __restrict__ scale_out) {
    __shared__ float smem[kNW];
    const int64_t row = blockIdx.x;
    float amax = 0.f;
    for (int64_t k = threadIdx.x; k < K; k += kThreads) amax = max_nonneg(amax, fabsf(wq_load<DT>(w, row * ldw + k)));
    const float m = block_max<kNW>(amax, smem);  // NaN if the row holds one, as torch's max
    const float s = wq_round<DT>(m / 127.f);
    if (threadIdx.x == 0) {
        if (DT == LLMQ_F32) reinterpret_cast<float*>(scale_out)[row] = s;
        else reinterpret_cast<uint16_t*>(scale_out)[row] = Lo<DT == LLMQ_F32 ? LLMQ_BF16 : DT>::from_f32(s);
    }
    for (int64_t k = threadIdx.x; k < K; k += kThreads) {
        const float t = wq_round<DT>(wq_load<DT>(w, row * ldw + k) / s);
        const float r = __builtin_rintf(t);
        q[row * K + k] = (t != t) ? (int8_t)0 : (int8_t)__builtin_amdgcn_fmed3f(r, -128.f, 127.f);
    }
}

}  // namespace
}  // namespace llmq

using namespace llmq;

extern "C" size_t llmq_quant_workspace_bytes(void) { return kMaxPartials * sizeof(float); }

extern "C" int llmq_quant_i8_per_token(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx,
                                       int8_t* q, void* scale, int scale_dtype, llmq_stream_t stream) {
    return llmq_quant_i8_per_token_floor(x, x_dtype, M, K, ldx, q, scale, scale_dtype, QP<MODE_I8>::floor_, stream);
}

extern "C" int llmq_quant_i8_per_token_floor(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx,
                                             int8_t* q, void* scale, int scale_dtype, float absmax_floor,
                                             llmq_stream_t stream) {
    if (!(absmax_floor >= 0.f)) return LLMQ_ERR_SHAPE;
    int rc = check_common(x, x_dtype, M, K, ldx, q);
    if (rc != LLMQ_OK) return rc;
    if (M == 0) return LLMQ_OK;
    if (!scale) return LLMQ_ERR_NULL;
    if (scale_dtype != x_dtype && scale_dtype != LLMQ_F32) return LLMQ_ERR_DTYPE;
    if (K == 0) return LLMQ_ERR_SHAPE;
    return dispatch_rows<MODE_I8, SCALE_ROW>(x, x_dtype, M, K, ldx, q, scale, scale_dtype, nullptr, 0, 0, absmax_floor,
                                             TensorAlpha{}, (hipStream_t)stream);
}

extern "C" int llmq_quant_i8_per_tensor(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx,
                                        int8_t* q, void* scale, int scale_dtype, void* workspace,
                                        size_t workspace_bytes, llmq_stream_t stream) {
    return llmq_quant_i8_per_tensor_floor(x, x_dtype, M, K, ldx, q, scale, scale_dtype, QP<MODE_I8>::floor_, workspace,
                                          workspace_bytes, stream);
}

extern "C" int llmq_quant_i8_per_tensor_floor(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx,
                                              int8_t* q, void* scale, int scale_dtype, float absmax_floor,
                                              void* workspace, size_t workspace_bytes, llmq_stream_t stream) {
    if (!(absmax_floor >= 0.f)) return LLMQ_ERR_SHAPE;
    int rc = check_common(x, x_dtype, M, K, ldx, q);
    if (rc != LLMQ_OK) return rc;
    if (!scale) return LLMQ_ERR_NULL;
    if (scale_dtype != x_dtype && scale_dtype != LLMQ_F32) return LLMQ_ERR_DTYPE;
    if (M == 0 || K == 0) return LLMQ_ERR_SHAPE;
    return per_tensor<MODE_I8>(x, x_dtype, M, K, ldx, q, scale, scale_dtype, workspace, workspace_bytes, absmax_floor,
                               TensorAlpha{}, (hipStream_t)stream);
}

extern "C" int llmq_quant_fp8_per_token(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx,
                                        uint8_t* q, float* scale, llmq_stream_t stream) {
    int rc = check_common(x, x_dtype, M, K, ldx, q);
    if (rc != LLMQ_OK) return rc;
    if (M == 0) return LLMQ_OK;
    if (!scale) return LLMQ_ERR_NULL;
    if (K == 0) return LLMQ_ERR_SHAPE;
    return dispatch_rows<MODE_F8, SCALE_ROW>(x, x_dtype, M, K, ldx, q, scale, LLMQ_F32, nullptr, 0, 0,
                                             QP<MODE_F8>::floor_, TensorAlpha{}, (hipStream_t)stream);
}

extern "C" int llmq_quant_fp8_per_tensor(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx,
                                         uint8_t* q, float* scale, void* workspace, size_t workspace_bytes,
                                         llmq_stream_t stream) {
    int rc = check_common(x, x_dtype, M, K, ldx, q);
    if (rc != LLMQ_OK) return rc;
    if (!scale) return LLMQ_ERR_NULL;
    if (M == 0 || K == 0) return LLMQ_ERR_SHAPE;
    return per_tensor<MODE_F8>(x, x_dtype, M, K, ldx, q, scale, LLMQ_F32, workspace, workspace_bytes,
                               QP<MODE_F8>::floor_, TensorAlpha{}, (hipStream_t)stream);
}

extern "C" int llmq_quant_per_tensor_alpha(int fp8, const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, void* q,
                                           float* scale, const float* w_scale, float* alpha, void* workspace,
                                           size_t workspace_bytes, llmq_stream_t stream) {
    int rc = check_common(x, x_dtype, M, K, ldx, q);
    if (rc != LLMQ_OK) return rc;
    if (!scale || !w_scale || !alpha) return LLMQ_ERR_NULL;
    if (M == 0 || K == 0) return LLMQ_ERR_SHAPE;
    const TensorAlpha ta{w_scale, alpha, fp8 ? 0 : 1};
    if (fp8)
        return per_tensor<MODE_F8>(x, x_dtype, M, K, ldx, q, scale, LLMQ_F32, workspace, workspace_bytes,
                                   QP<MODE_F8>::floor_, ta, (hipStream_t)stream);
    return per_tensor<MODE_I8>(x, x_dtype, M, K, ldx, q, scale, LLMQ_F32, workspace, workspace_bytes,
                               QP<MODE_I8>::floor_, ta, (hipStream_t)stream);
}

extern "C" int llmq_quant_fp8_static_alpha(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, uint8_t* q,
                                           const float* scale, int scale_is_f32_tensor, const float* w_scale, float* alpha,
                                           llmq_stream_t stream) {
    int rc = check_common(x, x_dtype, M, K, ldx, q);
    if (rc != LLMQ_OK) return rc;
    if (M == 0 || K == 0) return LLMQ_ERR_SHAPE;
    if (!scale || !w_scale || !alpha) return LLMQ_ERR_NULL;
    return dispatch_rows<MODE_F8, SCALE_STATIC>(x, x_dtype, M, K, ldx, q, nullptr, LLMQ_F32, scale, 1,
                                                scale_is_f32_tensor ? 1 : 0, 0.f, TensorAlpha{w_scale, alpha, 0},
                                                (hipStream_t)stream);
}

extern "C" int llmq_quant_fp8_static(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx,
                                     uint8_t* q, const float* scale, int scale_is_f32_tensor,
                                     llmq_stream_t stream) {
    int rc = check_common(x, x_dtype, M, K, ldx, q);
    if (rc != LLMQ_OK) return rc;
    if (M == 0 || K == 0) return LLMQ_OK;
    if (!scale) return LLMQ_ERR_NULL;
    return dispatch_rows<MODE_F8, SCALE_STATIC>(x, x_dtype, M, K, ldx, q, nullptr, LLMQ_F32, scale, 1,
                                                scale_is_f32_tensor ? 1 : 0, 0.f, TensorAlpha{}, (hipStream_t)stream);
}

extern "C" int llmq_quant_i8_weight_per_channel(const void* w, int w_dtype, int64_t N, int64_t K, int64_t ldw,
                                                int8_t* q, void* scale, llmq_stream_t stream) {
    if (w_dtype != LLMQ_BF16 && w_dtype != LLMQ_F16 && w_dtype != LLMQ_F32) return LLMQ_ERR_DTYPE;
    if (N < 0 || K < 0 || ldw < K || N > 0x7fffffffLL) return LLMQ_ERR_SHAPE;
    if (N == 0) return LLMQ_OK;
    if (K == 0) return LLMQ_ERR_SHAPE;
    if (!w || !q || !scale) return LLMQ_ERR_NULL;
    const dim3 grid((unsigned)N), block(kThreads);
    hipStream_t st = (hipStream_t)stream;
    if (w_dtype == LLMQ_BF16) hipLaunchKernelGGL((quant_weight_rows_kernel<LLMQ_BF16>), grid, block, 0, st, w, ldw, K, q, scale);
    else if (w_dtype == LLMQ_F16) hipLaunchKernelGGL((quant_weight_rows_kernel<LLMQ_F16>), grid, block, 0, st, w, ldw, K, q, scale);
    else hipLaunchKernelGGL((quant_weight_rows_kernel<LLMQ_F32>), grid, block, 0, st, w, ldw, K, q, scale);
    return launch_status();
}

extern "C" int llmq_rmsnorm(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const void* weight,
                            float eps, void* y, float* inv_rms, llmq_stream_t stream) {
    return rmsnorm_entry<-1>(x, x_dtype, M, K, ldx, weight, eps, y, nullptr, nullptr, LLMQ_F32, inv_rms,
                             (hipStream_t)stream);
}

extern "C" int llmq_rmsnorm_quant_i8_per_token(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx,
                                               const void* weight, float eps, void* y, int8_t* q, void* scale,
                                               int scale_dtype, float* inv_rms, llmq_stream_t stream) {
    return rmsnorm_entry<MODE_I8>(x, x_dtype, M, K, ldx, weight, eps, y, q, scale, scale_dtype, inv_rms,
                                  (hipStream_t)stream);
}

extern "C" int llmq_rmsnorm_quant_fp8_per_token(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx,
                                                const void* weight, float eps, void* y, uint8_t* q, float* scale,
                                                float* inv_rms, llmq_stream_t stream) {
    return rmsnorm_entry<MODE_F8>(x, x_dtype, M, K, ldx, weight, eps, y, q, scale, LLMQ_F32, inv_rms,
                                  (hipStream_t)stream);
}
