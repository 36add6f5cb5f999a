// W8A8 int8, FP8 (OCP e4m3fn / e5m2) and fp16 GEMMs: the planner (tile configuration, K split, few-token kernel,
// tail split) and the C entry points.  The tile kernels live in gemm_tile_impl.h and are instantiated per operand
// format in gemm_tile_*.hip; the few-token kernels in gemm_skinny.hip and gemm_rows.hip.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "gemm_rows.h"
#include "gemm_tile.h"
#include "llmq_common.h"

namespace llmq {

namespace {

// Tuning/diagnostic knob (llmq_gemm_force_plan): forces a tile configuration and K split.
thread_local int g_force_cfg = -1, g_force_splits = 1, g_force_dma = -1;  // per host thread; g_force_dma: 0 = register-staged loop only
bool plan_override(int& cfg, int& splits) {
    if (g_force_cfg < 0) return false;
    cfg = g_force_cfg;
    splits = g_force_splits;
    return true;
}

inline Plan skinny(int mt, int t, int nw, int64_t K) { return Plan{kSkinnyCfg + (t - 1) + (nw == 16 ? 4 : nw == 8 ? 2 : 0), 1, (int)K, mt}; }
inline int skinny_mt(int64_t M) { return M <= 16 ? 1 : (M <= 32 ? 2 : 4); }

// Up to 64 tokens in one block row: the streaming kernel without LDS staging.
bool skinny_plan(int64_t M, int64_t N, int64_t K, int& t, int& nw) {
    if (M > 64) return false;
    // Measured on the Qwen2-7B projections with the weights coming out of HBM, against the tile kernel (with and
    // without split K): ahead up to 16 tokens for every projection with N <= 8192 (8 tokens for a long K: every
    // wavefront re-reads the activations of its K run), and up to 32 tokens for a short K, where the tile kernel has
    // only N / 128 blocks to pull the weights with (o: 7.1 / 8.3 us against 14.0 / 13.1 at 17 / 32 tokens, qkv 9.4 /
    // 10.9 against 15.7 / 15.5); a narrow N keeps the lead to 64 tokens with 16 wavefronts along K (o: 11.3 against
    // 13.5 us).  For gate_up (N = 37888) the tile kernel already streams at 5.5 TB/s.
    if (N > 8192) return false;
    // Short K: more wavefronts along K would own a step or two each and wait for the block's reduction, so four and one
    // channel tile (4 / 8 / 16 wavefronts, us: 16 x 896 x 896 fp8 4.2 / 5.5 / 5.5, 40 x 896 x 1792 5.7 / 5.6 / 8.7,
    // 64 x 2048 x 896 4.9 / 6.5 / 6.7, int8 48 x 1152 x 896 4.6 / 5.9 / 9.2; at K = 3584 eight win, 5.3 against 5.8).
    if (K <= 2048 && N < 4096) {
        t = 1, nw = 4;
        return true;
    }
    if (K >= 8192) {
        if (M > 8) return false;
        t = 1, nw = 8;
        return true;
    }
    if (M <= 16) {
        if (N >= 4096) t = 2, nw = 4;
        else t = 1, nw = 8;
        return true;
    }
    if (M <= 32) {
        t = N >= 4096 ? 2 : 1, nw = 4;
        return true;
    }
    if (N < 4096) {
        t = 1, nw = 16;
        return true;
    }
    return false;
}

constexpr size_t kStaticScratchBytes = (size_t)32 << 20;  // the library's own scratch (llmq_gemm_w8a8_static)
inline size_t partials_bytes(const Plan& p, int64_t M, int64_t N) { return p.splits > 1 ? (size_t)p.splits * M * N * 4 : 0; }

// ---- Table plans: fewer than two rounds of 256x256 tiles and up to 20480 elements of K -------------------------------
constexpr int64_t kTableMaxK = 20480;  // elements
inline bool table_problem(int op, int64_t M, int64_t N, int64_t K) {  // K in bytes
    return M > (K % 128 ? 128 : 64) && (int64_t)cdiv(M, 256) * cdiv(N, 256) < 2 * kNumCu && K <= kTableMaxK * (op == 2 ? 2 : 1);
}

// More than 64 rows of whole 128-byte lines, more than 128 of others (whose K tail goes through registers).  Time (us) of a launch of x * 256
// blocks over `steps` times 64 bytes of K: each round of 256 blocks takes steps * step + fixed, a partly filled one with a share f
// of the CUs steps * step * (lo + (1 - lo) f) + fixed (fewer blocks share the supply and the clock is higher); the 64- and 32-row tiles
// share a CU: a block beside another takes `first` of its time.  Otherwise `first` is paid once.  The weights bound a launch from below (weights us per MB + base),
// outputs cost `out` us per MB, a K split the finishing launch and `partial` us per 8 MB of partial sums written and read (`past` on
// top for what exceeds the L2s' 32 MB).
// Fitted on an MI355X to every configuration x K split of 13 000 random problems (210 000 plans), for the time of the plan it picks: int8 and
// fp8 with weights out of HBM, fp16 with them in the Infinity Cache, where the dequantizer in front of it leaves them.  1.2-1.4 % behind
// the best plan in the mean (1.3-1.7 % on held-out problems); without the 128x128, 192x128 and 256x128 tiles of whole lines 5.7-6.7 %.  What
// those are for (us, best before / with them): fp8 1000 x 3584 x 3584 30.0 / 21.5 (128x128), 512 x 4608 x 3584 24.2 / 19.5, int8 1000 x
// 4608 x 3584 30.1 / 24.3 (192x128), fp8 512 x 37888 x 3584 87.8 / 84.4 (256x128).  (128x192 27.0 and 192x192 31.6 on the third, 256x320
// spills: not kept.)
struct TileCost { int cfg; double step, lo, fixed, first; };
struct FormatCost { double finish, partial, past, weights, base, out; TileCost tiles[7]; };
const FormatCost kCosts[3] = {
    {1.999, 1.651, 0.191, 0.090, 5.683, 0.074,  // int8
     {{4, 0.188, 0.697, 5.489, 1.278}, {5, 0.155, 0.780, 3.910, 0.538}, {6, 0.769, 0.730, 4.954, 2.081}, {7, 0.421, 0.600, 2.842, 3.415},
      {8, 0.259, 0.508, 3.676, 1.750}, {9, 0.334, 0.605, 3.239, 2.526}, {10, 0.404, 0.574, 4.578, 2.426}}},
    {2.721, 1.479, 0.100, 0.067, 5.194, 0.076,  // fp8
     {{4, 0.193, 0.602, 5.014, 0.906}, {5, 0.162, 0.823, 3.617, 0.429}, {6, 0.736, 0.861, 4.406, 2.222}, {7, 0.420, 0.592, 3.389, 2.941},
      {8, 0.252, 0.528, 3.087, 2.184}, {9, 0.326, 0.573, 3.406, 2.213}, {10, 0.381, 0.747, 3.471, 2.291}}},
    {1.780, 1.789, 0.000, 0.145, 1.300, 0.133,  // fp16
     {{4, 0.160, 0.599, 4.674, 0.970}, {5, 0.125, 0.721, 3.831, 0.729}, {6, 0.742, 0.674, 4.967, 1.522}, {7, 0.420, 0.522, 4.735, 2.094},
      {8, 0.255, 0.311, 4.284, 2.477}, {9, 0.327, 0.431, 4.315, 2.575}, {10, 0.411, 0.546, 4.554, 2.606}}}};

// Modelled time of configuration row `c` with K in sp splits of kps bytes; `limit` or more where it is certain to exceed that (the roots are
// most of a search).
double table_time(const FormatCost& f, const TileCost& c, int64_t M, int64_t N, int64_t K, int sp, int kps, double limit = 1e300) {
    const TileShape s = kShapes[c.cfg];
    const double run = kps / 64.0 * c.step, x = (double)((int64_t)cdiv(M, s.bm) * cdiv(N, s.bn) * sp) / kNumCu;
    const double full = std::floor(x), part = x - full, weights = (double)N * K * f.weights / 1e6 + f.base;
    double t;
    if (c.cfg <= 5) t = run * (x > 1 ? std::max(x, 1 + (std::ceil(x) - 1) * c.first) : c.lo + (1 - c.lo) * x) + c.fixed;
    else t = full * (run + c.fixed) + (part > 0 ? run * (c.lo + (1 - c.lo) * part) + c.fixed : 0) + c.first;
    double rest = (double)M * N * 2 * f.out / 1e6;
    if (sp > 1) {
        const double partials = (double)M * N * sp * 4;
        rest += f.finish + f.partial * partials * 2 / 8e6 + f.past * std::max(0.0, partials - 3.2e7) / 8e6;
    }
    const double least = (std::max(t, weights) + rest) * 0.999999;
    if (least >= limit) return least;
    const double t3 = t * t * t, w3 = weights * weights * weights;
    return std::cbrt(std::sqrt(t3 * t3 + w3 * w3)) + rest;
}
const FormatCost& costs_of(int op) { return kCosts[op == 1 ? 1 : op == 2 ? 2 : 0]; }

Plan table_plan(int op, int64_t M, int64_t N, int64_t K, size_t max_partials, double& best_t) {
    const FormatCost& f = costs_of(op);
    Plan best{8, 1, (int)K};
    best_t = 1e300;
    for (const TileCost& c : f.tiles) {
        for (int sp = 1; sp <= 16; sp += sp < 8 ? 1 : 2) {
            const size_t partials = sp > 1 ? (size_t)M * N * sp * 4 : 0;
            if (sp > 1 && (K / sp < 512 || partials > (size_t)256 << 20 || partials > max_partials)) break;
            const int kps = cdiv(cdiv(K, sp), 128) * 128;
            if (cdiv(K, kps) != sp) continue;
            const double t = table_time(f, c, M, N, K, sp, kps, best_t);
            if (t < best_t) best_t = t, best = Plan{c.cfg, sp, kps};
        }
    }
    return best;
}

// Few-token kernel in slabs of 16 * mt tokens: modelled us of a launch.  A wavefront's steps are a chain of load latencies that grows with the
// operands a step loads (`step` us per 16-row tile); blocks that share a CU slow each other down by `share`; a CU's loads move
// 1000 / `bytes` bytes per us; weights as in the table.  Fitted to 16 variants each of 8500 random problems of up to 512 tokens together with
// the tile plans of the same problems.  One launch instead of a K split and its finishing launch (us, rules alone / with slabs): int8 60 x
// 640 x 1664 7.4 / 4.4, 40 x 1152 x 6528 17.4 / 9.8, fp8 45 x 1152 x 1280 6.2 / 4.3, 200 x 512 x 3584 8.9 / 7.5.
struct SkinnyCost { double base, reduce, first, step, share, bytes, weights; };
const SkinnyCost kSkinnyCosts[2] = {{3.5187, 0.0362, 0.5059, 0.0416, 4.7137, 0.0274, 0.1709},   // int8
                                    {3.8676, 0.0165, 0.2335, 0.0591, 11.138, 0.0281, 0.1178}};  // fp8
double skinny_time(int op, int64_t M, int64_t N, int64_t K, int mt, int t, int nw) {
    const SkinnyCost& c = kSkinnyCosts[op == 1 ? 1 : 0];
    const double x = (double)((int64_t)cdiv(N, 16 * t) * cdiv(M, 16 * mt)) / kNumCu, steps = cdiv(cdiv(K, op == 1 ? 128 : 64), nw);
    const double chain = (steps * c.step * (t + mt) + c.first) * (1 + c.share * (std::ceil(x) - 1));
    const double supply = std::max(x, 1.0) * (t + mt) * 16 * K * c.bytes / 1e3, weights = (double)N * K * c.weights / 1e6;
    const double a = chain * chain, b = supply * supply, w = weights * weights;
    return c.base + c.reduce * mt * t * nw + std::sqrt(std::sqrt(a * a + b * b + w * w));
}
// Where slabs and tiles compete: up to 64 tokens and 8192 channels, 65-128 up to 2048, 129-256 up to 1024 (beyond, a tile plan was the fastest
// on 93-100 % of the problems); rows of whole 128-byte lines, as in the table.  Where the one-launch linear (linear_fused.hip) can take the
// problem, the rules of skinny_plan stand: it splits K as they do.
bool slab_problem(int op, int64_t M, int64_t N, int64_t K) {
    return op != 2 && (M > 16 || M * (K + 16) > 65280) && M <= 256 && K % 128 == 0 && K <= kTableMaxK && N <= (M <= 64 ? 8192 : M <= 128 ? 2048 : 1024);
}

// The plan among the configurations without the tiles of whole lines 8-10: what the table has to beat.  Fitted the same way to 311 000 plans of 12 600 random problems.
//   step      time per 64 bytes of K of a round of up to 256 blocks (a partly filled round takes as long as a full one)
//   fixed     prologue and epilogue of a round
//   ragged    factor on step where K % 128 != 0
//   shared    64- and 32-row tiles, which share a CU: past 256 blocks, time per 64 bytes of K and 256 blocks
//   finish, partial   finishing launch of a K split, and us per 8 MB of partial sums written and read
// A split whose partial sums exceed the 32 MB of the L2s must win by a tenth (without that margin 1.3 % of the problems end
// more than 5 % behind the rounds model, with it 0.6 %).
struct StagedCost { int cfg; double step, fixed, ragged, shared, finish, partial; };
Plan staged_plan(int op, int64_t M, int64_t N, int64_t K, size_t max_partials) {
    static const StagedCost kInt8F16[] = {{1, 0.707, 8.52, 1.248, 0, 3.91, 1.425},  // 256x256
                                          {2, 0.484, 8.53, 1.236, 0, 1.92, 1.319},  // 256x128
                                          {3, 0.275, 5.99, 1.298, 0, 3.77, 0.999}}; // 128x128
    static const StagedCost kFp8[] = {{1, 0.659, 10.33, 1.455, 0, 3.67, 1.630},
                                      {2, 0.629, 9.83, 1.113, 0, 1.94, 1.251},
                                      {3, 0.399, 6.36, 1.250, 0, 4.51, 0.446}};
    static const StagedCost kAll[] = {{4, 0.173, 3.60, 1.585, 0.225, 3.47, 1.522},  // 64x128
                                      {5, 0.167, 0.87, 1.400, 0.254, 3.77, 1.623},  // 32x128
                                      {7, 0.359, 6.97, 1.454, 0, 2.42, 1.867}};     // 128x256
    const bool ragged = K % 128 != 0;
    Plan best{1, 1, (int)K};
    double best_t = 1e300;
    for (int row = 0; row < 6; row++) {
        const StagedCost& c = row >= 3 ? kAll[row - 3] : (op == 1 ? kFp8 : kInt8F16)[row];
        const TileShape s = kShapes[c.cfg];
        const int64_t tiles = (int64_t)cdiv(M, s.bm) * cdiv(N, s.bn);
        const double step = c.step * (ragged ? c.ragged : 1.0), shared = c.shared * (ragged ? c.ragged : 1.0);
        for (int sp = 1; sp <= 16; sp += sp < 8 ? 1 : 2) {
            const size_t partials = sp > 1 ? (size_t)M * N * sp * 4 : 0;
            if (sp > 1 && (K / sp < 512 || partials > (size_t)256 << 20 || partials > max_partials)) break;
            const int kps = cdiv(cdiv(K, sp), s.bk) * s.bk;
            if (cdiv(K, kps) != sp) continue;
            const double steps = kps / 64.0, x = (double)tiles * sp / kNumCu, rounds = (double)cdiv(tiles * sp, kNumCu);
            double t = rounds * (steps * step + c.fixed);
            if (c.shared > 0 && x > 1) t = steps * std::max(shared * x, step) + c.fixed * 0.5 * (1 + rounds);
            if (sp > 1) t += c.finish + c.partial * partials * 2 / 8.0e6;
            if (partials > kStaticScratchBytes) t *= 1.1;
            if (t < best_t) best_t = t, best = Plan{c.cfg, sp, kps};
        }
    }
    return best;
}

// The rounds model, for up to 64 rows (128 with a ragged K), for grids of two rounds and more, and for a longer K:
// waves of blocks over the CUs x per-block MFMA time, with a floor from the bytes each block streams.
// The matrix cores take the same time per byte of K for int8, fp8 and fp16 (half the K elements at half the rate), so one
// table serves all three.  (Priced at twice the time per byte, fp16 was split five ways along K at 777 x 3584 x 18944: 138-140
// us with 55 MB of partial sums, against 132-136 us for the two-way split picked here.)
// fp8: the 64-byte K tiles have one MFMA sub-step there and keep the register-staged loop (measured ~20 % slower)
Plan rounds_plan(int64_t M, int64_t N, int64_t K, bool fp8) {
    int ocfg, osp;
    if (plan_override(ocfg, osp) && ocfg < 100) {
        const TileShape s = kShapes[ocfg < kNumShapes ? ocfg : kNumShapes - 1];
        const int kps = cdiv(cdiv(K, osp), s.bk) * s.bk;
        return Plan{ocfg < kNumShapes ? ocfg : kNumShapes - 1, cdiv(K, kps), kps};
    }
    // Cost model calibrated on MI355X (microseconds) with the direct-load kernels: a block needs t_tile per 64 bytes
    // of K plus a fixed prologue/epilogue cost; blocks execute in rounds over the 256 CUs (the small tiles are bound
    // by the CU's load path, so co-resident blocks share it and are not modelled as extra slots).  The chip is
    // power-limited under MFMA load: with a fraction f of the CUs busy a K tile takes (0.52 + 0.48 f) of its
    // full-chip time, so a partly filled round is cheaper than a full one.  Split-K adds a second kernel and the round
    // trip of the fp32/int32 partials.  Checked against a sweep of every configuration x K split at M = 128 / 512 /
    // 2048: the plan picked is within 1.5 % of the best measured one on average.
    struct Model { int cfg, per_cu; double t_tile, fixed; };
    static const Model kModels[] = {
        {1, 1, 0.88, 13.0},  // 256x256, 8 waves
        {2, 1, 0.60, 12.0},  // 256x128
        {3, 1, 0.27, 8.0},   // 128x128
        {4, 1, 0.17, 7.0},   // 64x128 (0.15 with its operands in the Infinity Cache; 0.17 is what it takes with weights out of HBM)
        {5, 1, 0.115, 4.1},  // 32x128: a chain of load latencies, the same however many CUs are busy
        {7, 1, 0.45, 8.0},   // 128x256, 8 waves
    };
    Plan best{1, 1, (int)K};
    double best_t = 1e300;
    for (const Model& md : kModels) {
        const TileShape s = kShapes[md.cfg];
        // small tiles are for small M; the 64-row tile also serves up to 1024 rows when 128x128 tiles
        // could not even fill the CUs once and K is short (measured: o and qkv at M = 512), and any M whose 64-row
        // grid fits the chip at once (fp8 2048 x 896 x 4864: 16.7 us against 28.5 with 128x256 tiles)
        if (M > 128 && md.cfg == 4 && (M > 1024 ? (int64_t)cdiv(M, 64) * cdiv(N, 128) > kNumCu
                                              : (int64_t)cdiv(M, 128) * cdiv(N, 128) >= 2 * kNumCu)) continue;
        if (md.cfg < 5 && M <= s.bm / 2) continue;            // mostly padding
        // 128x256 tiles are for grids that 256x256 tiles cannot fill twice over (measured: o / down at M = 2048,
        // gate_up at M = 512, qkv at M = 4096: 8-17 % ahead; with more tiles the big tile's lower operand traffic wins)
        if (md.cfg == 7 && (M <= 64 || (int64_t)cdiv(M, 256) * cdiv(N, 256) >= 2 * kNumCu)) continue;
        const int64_t tiles = (int64_t)cdiv(M, s.bm) * cdiv(N, s.bn);
        for (int sp = 1; sp <= 16; sp++) {
            if (sp > 1 && (K / sp < 512 || (int64_t)M * N * sp > (int64_t)64 << 20)) break;
            const int kps = cdiv(cdiv(K, sp), s.bk) * s.bk;
            const int eff_sp = cdiv(K, kps);
            if (eff_sp != sp) continue;
            const int64_t slots = (int64_t)kNumCu * md.per_cu, blocks = tiles * sp;
            // past 128 rows the 32-row tile is for grids that fit the chip at once (fp8, us, 64-row tile / 32-row tile:
            // 200 x 512 x 3584 12.7 / 9.0 with its K split, 256 x 896 x 4864 15.0 / 11.3, 1000 x 896 x 896 7.6 / 5.7);
            // beyond one round its operand traffic loses (1000 x 896 x 4864 as two splits 19.0 against 14.3 unsplit)
            if (md.cfg == 5 && M > 128 && blocks > slots) break;
            const int64_t full_rounds = blocks / slots, rest = blocks % slots;
            // fp8: the 64-byte K tiles run the slower register-staged loop; unsplit, config 1 is launched as the
            // 128-byte-tile config 6 (gemm_entry), which does not
            const double tt = md.t_tile * (fp8 && s.bk == 64 && !(md.cfg == 1 && sp == 1) ? 1.2 : 1.0);
            double t = full_rounds * (kps / 64.0 * tt + md.fixed);
            if (rest) t += kps / 64.0 * tt * (md.cfg == 5 ? 1.0 : 0.52 + 0.48 * (double)rest / slots) + md.fixed;
            // two 64-row blocks fit a CU side by side and share its load path: between one and two blocks per CU the
            // launch is one stretched round, not two (measured: 288 blocks of K = 3584 take 20 us, 224 take 14)
            if (md.cfg == 4 && blocks > slots && blocks <= 2 * slots) t = kps / 64.0 * tt * blocks / slots + md.fixed + 3.0;
            // the finishing launch, then the round trip of the partial sums.  Past the library's own scratch a split keeps the
            // dearer price it was calibrated with, so that llmq_gemm_w8a8_static goes on taking what it took
            if (sp > 1) t += ((size_t)M * N * sp * 4 > kStaticScratchBytes ? 5.0 : 3.5) + (double)M * N * sp * 8.0 / 8.0e6;
            if (t < best_t) { best_t = t; best = Plan{md.cfg, sp, kps}; }
        }
    }
    return best;
}

// The plan of a problem by operand format (0 int8, 1 fp8, 2 fp16; K in bytes).  kStaticInt8: int8 on the library's own scratch,
// which refuses what the rounds model splits past its size and runs the rest with a plan that fits.  With a ragged 8-bit K, whose
// price is the least certain, the other entry points stay within that size too where the rounds model does.
constexpr int kStaticInt8 = 3;
inline bool within_scratch(int op, int64_t K) { return op == kStaticInt8 || (op != 2 && K % 128 != 0); }

// The plan without slabs and without the table of the tiles of whole lines.  Its partial sums are what a size was first served with: a
// workspace of that size is still taken (gemm_entry) where the faster plan asks for more.
Plan rules_plan(int op, int64_t M, int64_t N, int64_t K) {
    int t, nw;
    if (op != 2 && skinny_plan(M, N, K, t, nw)) return skinny(skinny_mt(M), t, nw, K);
    if (M <= 128 || (int64_t)cdiv(M, 256) * cdiv(N, 256) >= 2 * kNumCu || K > kTableMaxK * (op == 2 ? 2 : 1)) return rounds_plan(M, N, K, op == 1);
    size_t most = SIZE_MAX;
    if (within_scratch(op, K)) {
        const Plan rounds = rounds_plan(M, N, K, op == 1);
        const bool fits = partials_bytes(rounds, M, N) <= kStaticScratchBytes;
        if (op == kStaticInt8 && !fits) return rounds;
        if (fits) most = kStaticScratchBytes;
    }
    return staged_plan(op, M, N, K, most);
}

// table_t: modelled time of the table's plan `table`, where one was searched
Plan tile_plan(int op, int64_t M, int64_t N, int64_t K, Plan& table, double& table_t) {
    const bool forced = g_force_cfg >= 0 && g_force_cfg < 100;
    if (forced || !table_problem(op, M, N, K)) return rounds_plan(M, N, K, op == 1);
    size_t most = SIZE_MAX;
    Plan old{};
    if (M <= 128 || within_scratch(op, K)) {
        old = rounds_plan(M, N, K, op == 1);
        const bool fits = partials_bytes(old, M, N) <= kStaticScratchBytes;
        if (op == kStaticInt8 && !fits) return old;
        if (fits && within_scratch(op, K)) most = kStaticScratchBytes;
    }
    table = table_plan(op, M, N, K, most, table_t);
    // The plan without the tiles of whole lines stays where it is of a configuration that the table prices (4-7; 2 and 3 give way to 8-10)
    // and the table's is not modelled as 6 % faster: of 2100 random problems of 300-8192 rows 4.4 % end more than 5 % behind it, without the
    // margin 7.1 %, at the same mean.
    if (M > 128) old = staged_plan(op, M, N, K, most);
    if (old.cfg == 1) old.cfg = 6, old.k_per_split = cdiv(old.k_per_split, 128) * 128;  // what config 1 is launched as
    for (const TileCost& c : costs_of(op).tiles)
        if (c.cfg == old.cfg && cdiv(K, old.k_per_split) == old.splits && table_t > 0.94 * table_time(costs_of(op), c, M, N, K, old.splits, old.k_per_split)) return old;
    return table;
}

// Long pieces of rows through LDS (gemm_rows.hip): modelled us.  `stage` is the time of a stage of a block that has its CU to itself; blocks beyond
// the first on a CU add `share` of it each; a CU's loads take `bytes` us per KB; weights `weights` us per MB.  Fitted to the time of each
// variant on 900 random problems of 1-64 tokens, int8 and fp8 alike, weights out of HBM (7-13 % standard deviation, 20 % for the 1024-byte pieces).
struct RowsCost { double base, stage, bytes, weights, share; };
const RowsCost kRowsCosts[kRowsMany] = {
    {2.8702, 0.2143, 0.0169, 0.1669, 1.5175},  // 1 x 1, 512 x 4
    {3.1549, 0.0033, 0.0128, 0.2272, 0.4290},  // 1 x 1, 1024 x 4
    {3.0883, 0.3853, 0.0000, 0.1691, 1.9517},  // 2 x 1, 512 x 4
    {2.8773, 0.3606, 0.0001, 0.2329, 1.0927},  // 1 x 2, 512 x 3
    {3.2079, 0.0016, 0.0121, 0.3053, 0.4101},  // 1 x 2, 1024 x 3
    {3.2159, 0.5002, 0.0000, 0.1909, 1.7175},  // 2 x 2, 512 x 3
    {2.8821, 0.7644, 0.0182, 0.2106, 0.6123},  // 2 x 2, 512 x 2
    {4.0008, 0.8345, 0.0001, 0.1795, 1.7072},  // 4 x 2, 512 x 3
    {3.4187, 0.4670, 0.0001, 0.2608, 1.6730},  // 1 x 3, 512 x 4
    {4.0452, 0.5548, 0.0001, 0.2358, 1.8744},  // 2 x 3, 512 x 3
    {3.3686, 0.4829, 0.0000, 0.3268, 1.7206},  // 1 x 4, 512 x 3
    {4.0328, 0.7390, 0.0000, 0.3058, 1.3016}};  // 2 x 4, 512 x 3
double rows_time(int v, int64_t N, int64_t K) {
    const RowsShape& s = kRowsShapes[v];
    const RowsCost& c = kRowsCosts[v];
    const double x = (double)cdiv(N, 16 * s.t) / kNumCu, stages = cdiv(K, s.seg);
    const double chain = stages * c.stage * (1 + c.share * (std::ceil(x) - 1)), supply = std::max(x, 1.0) * stages * 16 * (s.t + s.mt) * s.seg * c.bytes / 1e3;
    const double weights = (double)N * K * c.weights / 1e6, a = chain * chain, b = supply * supply, w = weights * weights;
    return c.base + std::sqrt(std::sqrt(a * a + b * b + w * w));
}
// Where it competes with the plan of tiles and gemm_skinny.hip, which takes `now` us as modelled: up to 64 tokens and not the shortest K, where
// a stage or two are all there is (us, now / rows: fp8 2 x 1024 x 1040 3.1 / 3.6, 2 x 576 x 3184 4.2 / 4.8, int8 18 x 3584 x 1744 4.5 /
// 4.8).
// `now` was fitted to more rows than these: for tiles it comes out at 0.7 of the measured time and at 0.55 where K ends inside a 128-byte line
// and the whole K tail goes through registers (36 x 10752 x 5792 28.8 / 24.5), for
// gemm_skinny.hip at 1.15.  With the factors below, of the 900 problems the half that moves makes the mean over all 11 % faster; 1 % of
// all end more than 5 % behind.
// Row lengths for which the same piece of the rows of a block falls on few memory channels: a few rows span a whole number of 32 KB, exactly or
// to 256 bytes.  Long pieces of many rows, all blocks at the same place of K, suffer more from it than the tiles' 128 bytes.
inline bool crowded_rows(int64_t K) {
    const auto near = [](int64_t v) { return (v + 256) % 32768 <= 512; };
    return K % 4096 == 0 || near(2 * K) || near(3 * K);
}
// Sizes at which the plan of tiles and gemm_skinny.hip (before) was measured ahead of this kernel (rows), in 10 000 random problems of 1-64 tokens that
// the lines of rows_variant give to it; us, before / rows.  With these the problems that end more than 3 % behind go from 819 to
// 181, more than 10 % from 262 to 7.
bool rows_behind(bool fp8, const Plan& plan, bool many, int64_t M, int64_t N, int64_t K) {
    const bool ragged = K % 128 != 0, tiles = plan.cfg < kSkinnyCfg;
    if (M > 16) {
        // three and four token tiles of few channels are few blocks over a long K (int8 61 x 960 x 8704 11.6 / 14.2, 50 x 512 x 9104 11.3 / 15.2; but fp8
        // 59 x 3472 x 7552 14.5 / 13.7), and over a short one wait for four wavefronts' sums (fp8 57 x 952 x 1920 4.4 / 5.1); many short ragged rows
        // (int8 49 x 9400 x 1984 12.6 / 14.4); the 4 KB stride (fp8 57 x 968 x 4096 7.1 / 8.3)
        if (M > 32) {
            if (tiles && K > 5632 && (M > 48 ? 3 : 4) * N < K && !(ragged && K <= 8192)) return true;
            if (plan.cfg == kSkinnyCfg && N <= 1280 && K <= 2048) return true;
            if (N > 8192 && K < 2560) return true;
            if (!ragged && N <= 1536 && K % 4096 == 0) return true;
        }
        // more than 256 tiles of 64 channels (int8 20 x 16808 x 1280 9.2 / 11.5, 29 x 24528 x 2000 16.4 / 18.8); 22 x 1080 x 15296 13.0 / 15.1
        return N > 16384 || (K > 10240 && 5 * N <= K);
    }
    if (many) {
        if (ragged) return false;
        // two stages or three of which the last is mostly empty, in more rounds than one (fp8 1 x 29256 x 1152 9.5 / 10.4, 2 x 25824 x 896 8.1 / 8.5;
        // but 2 x 25544 x 1024 8.7 / 8.3)
        if (N > 20480 && K < 1280 && K % 512) return true;
        // crowded rows, up to two groups a block: int8 2 x 14408 x 11008 33.1 / 38.9, 7 x 25576 x 8192 39.3 / 42.4, 4 x 22384 x 16384 66.5 / 80.0, 2 x 30896 x
        // 4096 24.9 / 28.1; fp8 8 x 8512 x 20480 37.9 / 42.7, 2 x 20544 x 16384 65.7 / 74.6; with three groups ahead again (int8 16 x 34104 x 8192 66.3 / 57.7)
        if (!crowded_rows(K) || N > 32768) return false;
        if (N <= 16384) return K > 10240 && !(fp8 && K >= 12288 && K <= 16512);
        if (fp8) return K == 16384 && N <= 24576;
        return K >= 16000 || 3 * K % 32768 <= 256 || (K == 8192 && N > 20480) || (K % 4096 == 0 && N > 24576);
    }
    if (ragged || tiles) return false;
    // eight or sixteen wavefronts along K that own no more than seven steps each (fp8 1 x 2760 x 3456 5.0 / 5.5, 4 x 3384 x 3456 5.4 / 5.7)
    if (K > 3136 && K <= 4096 && N < 4096 && ((M <= 2 && K < 4096) || (M <= 6 && N * K > 8800000))) return true;
    // crowded rows again (int8 1 x 3624 x 11008 11.1 / 13.1, 2 x 7984 x 16384 25.9 / 33.3, 3 x 8000 x 8192 14.7 / 16.7; fp8 2 x 7112 x 16384 26.0 / 30.2)
    if (K % 4096 != 0 && 3 * K % 32768 > 256) return false;
    return (M <= 3 && K >= 8192 && N > 2400 && N < 4096) || (M <= 8 && N > 6716 && (!fp8 || K >= 16384));
}
int rows_variant(int op, const Plan& plan, double now, int64_t M, int64_t N, int64_t K) {
    if (M > 64 || K <= (M <= 16 && N > 8192 ? 768 : 1024) || K > kTableMaxK) return -1;
    const int mt = cdiv(M, 16);
    // Many channels: blocks that go from one group of channels to the next, from where 64 channels a block are enough blocks.  3400 random problems
    // of up to 16 tokens, plan of tiles / this in the mean: 8193-16384 channels 1.20, 16385-24576 1.11, more 1.09; up to 8192 0.78.  16385-24576 channels
    // make one to one and a half groups of 64 a CU, so groups of 32 there, three a block: 1.10 against 1.08.
    // Up to 20480 of these the tiles of 128 channels fill the chip in one round and keep the shorter K (14 x 17920 x 4096 13.6 / 14.8, 4 x 19184 x 2432
    // 9.7 / 10.4; 2 x 18432 x 11904 48 / 42).
    const bool ragged = K % 128 != 0, tiles = plan.cfg < kSkinnyCfg;
    if (mt == 1 && N > 8192 && (N <= 16384 || N > 20480 || ragged || K >= 8192))
        return rows_behind(op == 1, plan, true, M, N, K) ? -1 : N > 16384 && N <= 24576 ? kRowsMany + 1 : kRowsMany;
    double factor = 0.95;
    if (mt > 1) {
        if (ragged && K < 2048 && N < 4096) return -1;
        if (tiles) factor = ragged ? 1.35 : 1.15;
    } else if (tiles) {
        if (N > 8192) return -1;
        factor = ragged ? 1.9 : 1.15;
    } else {
        if (N < 4096 ? K <= (ragged ? 4095 : 2048) : ragged && K < 1792) return -1;
        if (ragged && N * K > 40000000) return -1;  // (int8 3 x 2944 x 18608 12.9 / 15.6)
    }
    if (rows_behind(op == 1, plan, false, M, N, K)) return -1;
    double best = now * factor;
    int variant = -1;
    for (int v = 0; v < kRowsMany; v++)
        if (kRowsShapes[v].mt == mt) {
            const double t = rows_time(v, N, K);
            if (t < best) best = t, variant = v;
        }
    return variant;
}
inline Plan rows(int variant, int64_t K) { return Plan{kRowsCfg + variant, 1, (int)K}; }

Plan tiles_or_skinny_plan(int op, int64_t M, int64_t N, int64_t K) {
    int t, nw;
    if (g_force_cfg >= kRowsCfg && op != 2 && M <= 16 * kRowsShapes[g_force_cfg - kRowsCfg].mt) return rows(g_force_cfg - kRowsCfg, K);
    if (g_force_cfg >= kSkinnyCfg && g_force_cfg < kRowsCfg && op != 2) {  // forced few-token variant: 16, 32 or 64 as its split are the tokens of a slab
        const int slab = g_force_splits;
        if (slab == 16 || slab == 32 || slab == 64) return Plan{g_force_cfg, 1, (int)K, slab / 16};
        if (M <= 64) return Plan{g_force_cfg, 1, (int)K, skinny_mt(M)};
    }
    const bool few = g_force_cfg < 0 && op != 2 && skinny_plan(M, N, K, t, nw);
    Plan best{};
    double best_t = -1;
    const Plan plan = few ? skinny(skinny_mt(M), t, nw, K) : tile_plan(op, M, N, K, best, best_t);
    if (g_force_cfg >= 0 || !slab_problem(op, M, N, K)) return plan;
    if (op == kStaticInt8 && partials_bytes(plan, M, N) > kStaticScratchBytes) return plan;  // refused, as before
    // Sixteen wavefronts along a K of a few thousand in one block row: measured best there (slabs 8 % slower in the mean at 33-64 tokens of
    // more than 3000 channels, level at 2049-3000; 18-43 % faster with fewer channels, 40 % with a longer K).
    if (few && M > 32 && N > 2048 && K > 2048 && K <= 4096) return plan;
    // The plan of the rules stays unless another is modelled as clearly faster.
    double now = 1e300;
    if (few) now = skinny_time(op, M, N, K, skinny_mt(M), t, nw);
    else
        for (const TileCost& c : costs_of(op).tiles)
            if (c.cfg == plan.cfg) now = table_time(costs_of(op), c, M, N, K, plan.splits, plan.k_per_split);
    if (best_t < 0) best = table_plan(op, M, N, K, op == kStaticInt8 ? kStaticScratchBytes : SIZE_MAX, best_t);
    // Slabs of 16 or 32 tokens with four wavefronts along K: of 3 million random problems one picks another number of wavefronts, none 64 tokens.
    for (int mt = 1; mt <= (M > 16 ? 2 : 1); mt++)
        for (t = 1; t <= 2; t++) {
            const double s = skinny_time(op, M, N, K, mt, t, 4);
            if (s < best_t) best_t = s, best = skinny(mt, t, 4, K);
        }
    // By a tenth (2.1 % of 8600 random problems here end more than 5 % behind the rules, against 4.0 % without a margin, for 1.113 of the
    // 1.118 in the mean), by more where the rules pick the few-token kernel themselves: most of those were such problems with a short K.
    // A K split gives way to one launch of slabs at the same modelled time: the gap before its finishing launch is not in the model.
    const bool one_launch = best.cfg >= kSkinnyCfg && plan.splits > 1;
    return best_t < (few ? (K <= 1024 ? 0.75 : 0.85) : one_launch ? 1.0 : 0.9) * now ? best : plan;
}

Plan make_plan(int op, int64_t M, int64_t N, int64_t K) {
    const Plan plan = tiles_or_skinny_plan(op, M, N, K);
    if (g_force_cfg >= 0 || op == 2 || M > 64) return plan;
    if (op == kStaticInt8 && partials_bytes(plan, M, N) > kStaticScratchBytes) return plan;  // refused, as before
    double now = 1e300;
    if (plan.cfg >= kSkinnyCfg) now = skinny_time(op, M, N, K, plan.mt, 1 + ((plan.cfg - kSkinnyCfg) & 1), 4 << ((plan.cfg - kSkinnyCfg) >> 1));
    else
        for (const TileCost& c : costs_of(op).tiles)
            if (c.cfg == plan.cfg) now = table_time(costs_of(op), c, M, N, K, plan.splits, plan.k_per_split);
    const int variant = rows_variant(op, plan, now, M, N, K);
    return variant < 0 ? plan : rows(variant, K);
}

// Searching a plan takes microseconds of host time and a call needs it for its workspace and for its launch, so each host
// thread remembers the last plans it made (a pure function of sizes and format; a forced plan is not remembered).
constexpr int kCachedSizes = 64;
inline int size_slot(int64_t M, int64_t N, int64_t K, int op) { return ((uint64_t)(M * 31 + N * 17 + K * 7 + op) * 0x9E3779B97F4A7C15ull) >> 58; }
Plan plan_for(int op, int64_t M, int64_t N, int64_t K) {
    if (g_force_cfg >= 0) return make_plan(op, M, N, K);
    struct Entry { int64_t M, N, K; int op; Plan plan; };
    static thread_local Entry cache[kCachedSizes] = {};
    Entry& e = cache[size_slot(M, N, K, op)];
    if (e.M != M || e.N != N || e.K != K || e.op != op) e = Entry{M, N, K, op, make_plan(op, M, N, K)};
    return e.plan;
}

// op: 0 int8, 1 fp8 (a_format picks the A format), 2 fp16 (K, lda, ldb in bytes, i.e. twice the element counts)
// out_scale (device scalar, may be null): out is fp32 [M, N] holding the out_dtype result after a round trip through
// e4m3fn on that scale (tile kernel's general epilogue; no tail split)
int gemm_entry(int op, int a_format, const uint8_t* A, int64_t lda, const uint8_t* B, int64_t ldb,
               const float* a_scale, const float* w_scale, float alpha, const float* alpha_dev, const void* bias,
               int bias_dtype, float beta, void* out, int out_dtype, int64_t ldo, int64_t M, int64_t N, int64_t K,
               void* acc_dump, void* ws, size_t ws_bytes, hipStream_t st, const float* out_scale = nullptr,
               bool static_scratch = false) {
    const bool fp8 = op == 1;
    if (M < 0 || N < 0 || K < 0) return LLMQ_ERR_SHAPE;
    if (M == 0 || N == 0) return LLMQ_OK;
    if (!A || !B || !out) return LLMQ_ERR_NULL;
    if (K == 0 || (K & 15) || (lda & 15) || (ldb & 15) || lda < K || ldb < K || ldo < N) return LLMQ_ERR_SHAPE;
    if (M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL || lda >= (1 << 22) || ldb >= (1 << 22)) return LLMQ_ERR_SHAPE;
    if (out_dtype != LLMQ_BF16 && out_dtype != LLMQ_F16) return LLMQ_ERR_DTYPE;
    if (bias && bias_dtype != LLMQ_BF16 && bias_dtype != LLMQ_F16 && bias_dtype != LLMQ_F32) return LLMQ_ERR_DTYPE;
    if (fp8 && a_format != LLMQ_E4M3 && a_format != LLMQ_E5M2) return LLMQ_ERR_DTYPE;
    if (!aligned16(A) || !aligned16(B)) return LLMQ_ERR_ALIGN;
    auto fits = [&](const Plan& pl) { return pl.splits == 1 || (ws && ws_bytes >= partials_bytes(pl, M, N)); };
    const int planned_op = static_scratch ? kStaticInt8 : op;
    Plan p = plan_for(planned_op, M, N, K);
    if (!fits(p) && g_force_cfg < 0) p = rules_plan(planned_op, M, N, K);  // the caller kept the size that was enough for these
    if (!fits(p)) return LLMQ_ERR_WORKSPACE;
    if (p.cfg >= kSkinnyCfg) {  // both few-token kernels
        const SkinnyEpilogue sep{a_scale, w_scale, alpha_dev, bias, alpha, beta, bias_dtype, out_dtype, out_scale};
        if (p.cfg >= kRowsCfg)
            return launch_gemm_rows(fp8, a_format == LLMQ_E5M2 ? 1 : 0, p.cfg - kRowsCfg, A, lda, B, ldb, (int)M, (int)N, (int)K, sep, out, ldo, acc_dump, st);
        const int v = p.cfg - kSkinnyCfg;
        return launch_gemm_skinny(fp8, a_format == LLMQ_E5M2 ? 1 : 0, p.mt, 1 + (v & 1), 4 << (v >> 1), A, lda, B, ldb, (int)M, (int)N,
                                  (int)K, sep, out, ldo, acc_dump, st);
    }
    // The 256x256 tile runs with 128-byte K tiles (half the barriers, whole lines per row) where the split allows it.
    if (g_force_cfg < 0 && p.cfg == 1 && (p.splits == 1 || p.k_per_split % 128 == 0)) {
        p.cfg = 6;
        if (p.splits == 1) p.k_per_split = cdiv(K, 128) * 128;
    }
    auto run = [&](const Plan& pl, const uint8_t* Bp, const float* wsc, const void* bs, void* o, int64_t n) {
        Epilogue ep{a_scale, wsc, alpha_dev, bs, alpha, beta, bias_dtype, out_dtype, out_scale};
        const bool dma = g_force_dma != 0;
        if (op == 2) return launch_gemm_f16(A, lda, Bp, ldb, (int)M, (int)n, (int)K, pl, ep, o, ldo, acc_dump, ws, dma, st);
        if (!fp8) return launch_gemm_i8(A, lda, Bp, ldb, (int)M, (int)n, (int)K, pl, ep, o, ldo, acc_dump, ws, dma, st);
        if (a_format == LLMQ_E4M3)
            return launch_gemm_fp8_e4m3(A, lda, Bp, ldb, (int)M, (int)n, (int)K, pl, ep, o, ldo, acc_dump, ws, dma, st);
        return launch_gemm_fp8_e5m2(A, lda, Bp, ldb, (int)M, (int)n, (int)K, pl, ep, o, ldo, acc_dump, ws, dma, st);
    };
    // Tail split.  When the 256x256 grid ends in a round that fills at most 5/8 of the CUs, the channels are cut at a
    // whole number of rounds: the first part keeps the big tiles and ends with every CU busy, the rest runs as one
    // round of 128x256 tiles (twice the blocks, half the time each).  Measured: 8192 x 4608 x 3584 (2.25 rounds)
    // and 8192 x 37888 x 3584 (18.5 rounds).
    if (g_force_cfg < 0 && p.cfg == 6 && p.splits == 1 && !acc_dump && !out_scale) {
        const int64_t tm = cdiv(M, 256), tn = cdiv(N, 256), tiles = tm * tn, tail = tiles % kNumCu, full = tiles - tail;
        if (full >= kNumCu && tail > 0 && tail <= 160 && full % tm == 0) {
            const int64_t n1 = full / tm * 256, n2 = N - n1;
            if (n2 > 0 && (int64_t)cdiv(M, 128) * cdiv(n2, 256) <= kNumCu) {
                const int rc = run(p, B, w_scale, bias, out, n1);
                if (rc != LLMQ_OK) return rc;
                const int64_t be = bias_dtype == LLMQ_F32 ? 4 : 2;
                return run(Plan{7, 1, cdiv(K, 128) * 128}, B + n1 * ldb, w_scale ? w_scale + n1 : nullptr,
                           bias ? static_cast<const uint8_t*>(bias) + n1 * be : nullptr, static_cast<uint8_t*>(out) + n1 * 2, n2);
            }
        }
    }
    return run(p, B, w_scale, bias, out, N);
}

// ---- scratch owned by the library, for the entry point that takes no workspace ---------------------
// One copy of this array exists on every GPU the library is loaded on, for the life of the process.
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
// `scratch` is a host-side stand-in for the symbol, not a device address: the address of each GPU's copy
// is looked up once per device and only that pointer is ever handed to a kernel.
void* g_scratch_ptr[64] = {};

int static_scratch(void** out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return LLMQ_ERR_LAUNCH;
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return LLMQ_ERR_LAUNCH;
        g_scratch_ptr[dev] = p;  // benign if two threads race here: both store the same address
    }
    *out = g_scratch_ptr[dev];
    return LLMQ_OK;
}

}  // namespace
}  // namespace llmq

using namespace llmq;

extern "C" size_t llmq_gemm_static_scratch_bytes(void) { return kStaticScratchBytes; }

extern "C" int llmq_gemm_w8a8_static(const int8_t* A, int64_t lda, const int8_t* B, int64_t ldb, const float* a_scale,
                                     const float* w_scale, float alpha, const float* alpha_dev, const void* bias,
                                     int bias_dtype, float beta, void* out, int out_dtype, int64_t ldo, int64_t M,
                                     int64_t N, int64_t K, llmq_stream_t stream) {
    void* ws = nullptr;
    int rc = static_scratch(&ws);
    if (rc != LLMQ_OK) return rc;
    // The common entry validates the arguments first and then checks the partial sums of the plan it is about to
    // launch against the size it is given: a plan that does not fit the array is refused there, before any launch.
    rc = gemm_entry(0, 0, (const uint8_t*)A, lda, (const uint8_t*)B, ldb, a_scale, w_scale, alpha, alpha_dev, bias,
                    bias_dtype, beta, out, out_dtype, ldo, M, N, K, nullptr, ws, kStaticScratchBytes,
                    (hipStream_t)stream, nullptr, true);
    return rc == LLMQ_ERR_WORKSPACE ? LLMQ_ERR_SCRATCH : rc;
}

extern "C" int llmq_gemm_force_plan(int cfg, int splits) {
    int dma = -1;
    if (cfg >= 0 && cfg < 100 && (cfg & 64)) dma = 0, cfg &= ~64;
    if ((cfg >= kNumShapes && (cfg < kSkinnyCfg || (cfg > kSkinnyCfg + 5 && cfg < kRowsCfg) || cfg >= kRowsCfg + kRowsVariants)) || splits < 1 || splits > 64) return LLMQ_ERR_SHAPE;
    g_force_dma = dma;
    g_force_cfg = cfg;
    g_force_splits = splits;
    return LLMQ_OK;
}

extern "C" int llmq_gemm_num_configs(void) { return kNumShapes; }

// Sizes (K in bytes) of which a call can be taken; the planners count in 32 bits.
static bool plannable(int64_t M, int64_t N, int64_t K) { return M > 0 && N > 0 && K > 0 && M <= 0x7fffffffLL && N <= 0x7fffffffLL && K < (1 << 22); }

extern "C" int llmq_gemm_planned_config(int fp8, int64_t M, int64_t N, int64_t K) {
    return !plannable(M, N, K) || K % 16 ? LLMQ_ERR_SHAPE : plan_for(fp8 ? 1 : 0, M, N, K).cfg;
}

namespace {
// what the plan that a call of this size runs splits into: a lookup once the size is planned
size_t planned_bytes(int op, int64_t M, int64_t N, int64_t K) {
    return !plannable(M, N, K) ? 0 : partials_bytes(plan_for(op, M, N, K), M, N);
}
}  // namespace

extern "C" size_t llmq_gemm_w8a8_workspace_bytes(int64_t M, int64_t N, int64_t K) { return planned_bytes(0, M, N, K); }
extern "C" size_t llmq_gemm_fp8_workspace_bytes(int64_t M, int64_t N, int64_t K) { return planned_bytes(1, M, N, K); }
// For both formats, and no less than what the plans of the rules split: a figure that was enough for every plan this library had for a size.
extern "C" size_t llmq_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (g_force_cfg >= 0 || !plannable(M, N, K)) return std::max(planned_bytes(0, M, N, K), planned_bytes(1, M, N, K));
    struct Entry { int64_t M, N, K; size_t bytes; };
    static thread_local Entry cache[kCachedSizes] = {};
    Entry& e = cache[size_slot(M, N, K, 0)];
    if (e.M != M || e.N != N || e.K != K) {
        size_t most = 0;
        for (int op = 0; op < 2; op++)
            most = std::max({most, planned_bytes(op, M, N, K), partials_bytes(rules_plan(op, M, N, K), M, N)});
        e = Entry{M, N, K, most};
    }
    return e.bytes;
}

extern "C" int llmq_gemm_w8a8(const int8_t* A, int64_t lda, const int8_t* B, int64_t ldb, const float* a_scale,
                              const float* w_scale, float alpha, const float* alpha_dev, const void* bias,
                              int bias_dtype, float beta, void* out, int out_dtype, int64_t ldo, int64_t M, int64_t N,
                              int64_t K, int32_t* acc_dump, void* workspace, size_t workspace_bytes,
                              llmq_stream_t stream) {
    return gemm_entry(0, 0, (const uint8_t*)A, lda, (const uint8_t*)B, ldb, a_scale, w_scale, alpha, alpha_dev,
                      bias, bias_dtype, beta, out, out_dtype, ldo, M, N, K, acc_dump, workspace, workspace_bytes,
                      (hipStream_t)stream);
}

extern "C" int llmq_gemm_fp8(const uint8_t* A, int a_format, int64_t lda, const uint8_t* B, int64_t ldb,
                             const float* a_scale, const float* w_scale, float alpha, const float* alpha_dev,
                             const void* bias, int bias_dtype, float beta, void* out, int out_dtype, int64_t ldo,
                             int64_t M, int64_t N, int64_t K, float* acc_dump, void* workspace,
                             size_t workspace_bytes, llmq_stream_t stream) {
    return gemm_entry(1, a_format, A, lda, B, ldb, a_scale, w_scale, alpha, alpha_dev, bias, bias_dtype, beta, out,
                      out_dtype, ldo, M, N, K, acc_dump, workspace, workspace_bytes, (hipStream_t)stream);
}

extern "C" int llmq_gemm_fp8_quantized_output(const uint8_t* A, int a_format, int64_t lda, const uint8_t* B, int64_t ldb,
                                              const float* a_scale, const float* w_scale, float alpha,
                                              const float* alpha_dev, const void* bias, int bias_dtype, float beta,
                                              const float* out_scale, float* out, int inter_dtype, int64_t ldo, int64_t M,
                                              int64_t N, int64_t K, void* workspace, size_t workspace_bytes,
                                              llmq_stream_t stream) {
    if (!out_scale) return LLMQ_ERR_NULL;
    return gemm_entry(1, a_format, A, lda, B, ldb, a_scale, w_scale, alpha, alpha_dev, bias, bias_dtype, beta, out,
                      inter_dtype, ldo, M, N, K, nullptr, workspace, workspace_bytes, (hipStream_t)stream, out_scale);
}

extern "C" size_t llmq_gemm_fp8_quantized_output_workspace_bytes(int64_t M, int64_t N, int64_t K) { return planned_bytes(1, M, N, K); }

extern "C" size_t llmq_gemm_f16_workspace_bytes(int64_t M, int64_t N, int64_t K) { return planned_bytes(2, M, N, 2 * K); }

extern "C" int llmq_gemm_f16(const void* A, int64_t lda, const void* B, int64_t ldb, float alpha, const void* bias,
                             int bias_dtype, float beta, void* out, int out_dtype, int64_t ldo, int64_t M, int64_t N,
                             int64_t K, float* acc_dump, void* workspace, size_t workspace_bytes, llmq_stream_t stream) {
    if (K < 0 || (K & 7) || (lda & 7) || (ldb & 7)) return LLMQ_ERR_SHAPE;  // 16-byte pieces of fp16
    return gemm_entry(2, 0, (const uint8_t*)A, 2 * lda, (const uint8_t*)B, 2 * ldb, nullptr, nullptr, alpha, nullptr, bias,
                      bias_dtype, beta, out, out_dtype, ldo, M, N, 2 * K, acc_dump, workspace, workspace_bytes,
                      (hipStream_t)stream);
}
