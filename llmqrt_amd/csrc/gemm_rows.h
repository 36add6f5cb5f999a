// Few-token GEMMs in one launch without a workspace (gemm_skinny.hip: operands straight into registers; gemm_rows.hip: long pieces of
// rows through LDS), dispatched from gemm_mfma.hip.
#pragma once
#include "llmq_common.h"

namespace llmq {

struct SkinnyEpilogue {
    const float* a_scale;    // [M] or null
    const float* w_scale;    // [N] or null
    const float* alpha_dev;  // device scalar or null
    const void* bias;        // [N] or null
    float alpha, beta;
    int bias_dtype, out_dtype;
    const float* out_scale;  // device scalar or null: out is fp32 and holds the value after a round trip through e4m3fn on it
};

// mt: 16-token tiles per block (1 | 2 | 4), t: 16-channel tiles per wavefront (1 | 2), nw: wavefronts per block (4 | 8 | 16; 4 | 8 for
// mt = 4 and t = 2); a_format: 0 e4m3, 1 e5m2 (fp8 only)
int launch_gemm_skinny(bool fp8, int a_format, int mt, int t, int nw, const uint8_t* A, int64_t lda, const uint8_t* B, int64_t ldb,
                       int M, int N, int K, const SkinnyEpilogue& ep, void* out, int64_t ldo, void* acc_dump, hipStream_t st);

// Variants of gemm_rows.hip: t, mt 16-channel / 16-token tiles of a block, seg bytes of every row per stage, ns stages in LDS; many: a block
// takes several groups of channels.
#define LLMQ_ROWS_VARIANTS(V)                                                                                                          \
    V(0, 1, 1, 512, 4, false) V(1, 1, 1, 1024, 4, false) V(2, 2, 1, 512, 4, false) V(3, 1, 2, 512, 3, false) V(4, 1, 2, 1024, 3, false) \
    V(5, 2, 2, 512, 3, false) V(6, 2, 2, 512, 2, false) V(7, 4, 2, 512, 3, false) V(8, 1, 3, 512, 4, false) V(9, 2, 3, 512, 3, false)   \
    V(10, 1, 4, 512, 3, false) V(11, 2, 4, 512, 3, false) V(12, 4, 1, 512, 3, true) \
    V(13, 2, 1, 512, 3, true)
constexpr int kRowsVariants = 14, kRowsMany = 12;
struct RowsShape { int t, mt, seg, ns; };
constexpr RowsShape kRowsShapes[kRowsVariants] = {
#define LLMQ_ROWS_SHAPE(I, T, MT, SEG, NS, MANY) {T, MT, SEG, NS},
    LLMQ_ROWS_VARIANTS(LLMQ_ROWS_SHAPE)
#undef LLMQ_ROWS_SHAPE
};

// M <= 16 * kRowsShapes[variant].mt; anything else is refused
int launch_gemm_rows(bool fp8, int a_format, int variant, const uint8_t* A, int64_t lda, const uint8_t* B, int64_t ldb, int M, int N, int K,
                     const SkinnyEpilogue& ep, void* out, int64_t ldo, void* acc_dump, hipStream_t st);

}  // namespace llmq
