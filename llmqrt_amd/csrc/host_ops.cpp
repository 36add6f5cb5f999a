// Host side of the quantized modules' forward passes: one native call per module and token batch.
//
// A decode step of a layer is a handful of kernels of 3-30 us; driven from Python (argument checks, tensor allocations and
// ctypes calls of 20 arguments per kernel) the host needed 25-45 us per Linear and the GPU waited for it.  Each function
// here takes the module's tensors, checks the layout the kernels want, allocates from torch's caching allocator, and
// launches through the C ABI of libllmq_gfx950.so on the current stream.  It computes nothing and keeps no answer; an
// input outside the layout (strided rows, other dtypes, a tensor on another device, ...) returns None, and the caller's
// general Python path takes over, with its conversions and its error messages.
//
// Scratch comes from the caching allocator per call (stream-ordered, so safe with any number of threads and streams).
// The one thing kept between calls is the arrival counters of the few-token AWQ kernel: 512 KiB per device and stream,
// zeroed once and left zero by every call; calls on one stream run in order, calls on two streams use two sets, a capture
// has a set of its own per stream.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <mutex>
#include <optional>
#include <stdexcept>
#include <string>
#include <unordered_map>

#include "llmq.h"

namespace {

using at::Tensor;

void check(int status, const char* what) {
    if (status != LLMQ_OK)
        throw std::runtime_error(std::string(what) + ": " + llmq_status_string(status) + " (llmq status " +
                                 std::to_string(status) + ")");
}

bool is16(at::ScalarType t) { return t == at::kBFloat16 || t == at::kHalf; }
int code(at::ScalarType t) { return t == at::kBFloat16 ? LLMQ_BF16 : t == at::kHalf ? LLMQ_F16 : LLMQ_F32; }
bool aligned(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0; }
bool plain_on(const Tensor& t, const at::Device& dev) { return t.layout() == at::kStrided && t.device() == dev && t.is_contiguous(); }

Tensor make(at::IntArrayRef size, at::ScalarType dtype, const at::Device& dev) {
    return Tensor(at::detail::empty_cuda(size, dtype, dev, std::nullopt));
}

int64_t round16(int64_t n) { return (n + 15) & ~(int64_t)15; }

// Activations as [M, K] rows: contiguous, 16-byte aligned, at least one row.
struct Rows {
    int64_t M = 0, K = 0;
    bool ok = false;
};
Rows rows_of(const Tensor& x) {
    Rows r;
    if (!x.defined() || !x.is_cuda() || x.layout() != at::kStrided || x.dim() < 1 || x.numel() == 0 || !x.is_contiguous() ||
        !aligned(x))
        return r;
    r.K = x.size(-1);
    r.M = x.numel() / r.K;
    r.ok = true;
    return r;
}

at::DimVector out_size(const Tensor& x, int64_t n) {
    at::DimVector s(x.sizes().begin(), x.sizes().end());
    s.back() = n;
    return s;
}

struct Launch {
    c10::DeviceGuard guard;
    llmq_stream_t stream;
    explicit Launch(const at::Device& dev) : guard(dev), stream(c10::hip::getCurrentHIPStream(dev.index()).stream()) {}
};
// Whether a linear runs in one launch: where that is ahead on the GPU, and where the saved launch is worth more to the host than it costs the
// GPU, which no replayed graph gets back.  The current device is the stream's (Launch).
bool one_launch(int kind, int64_t M, int64_t N, int64_t K) {
    return llmq_linear_one_launch_preferred(kind, M, N, K) &&
           (llmq_linear_one_launch_ahead(kind, M, N, K) || c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None);
}

// The weight side of an 8-bit Linear: [N, K] bytes, K % 16 == 0.
bool weight_ok(const Tensor& w, at::ScalarType dtype, const at::Device& dev, int64_t K) {
    return w.defined() && w.scalar_type() == dtype && w.dim() == 2 && w.size(1) == K && w.size(0) > 0 && K % 16 == 0 &&
           plain_on(w, dev) && aligned(w);
}
bool scale_ok(const Tensor& s, const at::Device& dev, int64_t n) {
    return s.defined() && s.scalar_type() == at::kFloat && s.numel() == n && plain_on(s, dev);
}
bool bias_ok(const std::optional<Tensor>& b, const at::Device& dev, int64_t N) {
    return !b || (b->dim() == 1 && b->numel() == N && plain_on(*b, dev));
}
const void* ptr(const std::optional<Tensor>& t) { return t ? t->data_ptr() : nullptr; }

// GEMM operands that are the same for int8 and fp8
struct Gemm {
    bool fp8;
    const void* q;
    const Tensor& w;
    const float *a_scale, *w_scale, *alpha;
    const std::optional<Tensor>& bias;
    int64_t M, K;
};
void gemm(const Gemm& g, Tensor& out, at::ScalarType out_dtype, const Launch& l) {
    const int64_t N = g.w.size(0);
    const int64_t ws_bytes = (int64_t)(g.fp8 ? llmq_gemm_fp8_workspace_bytes : llmq_gemm_w8a8_workspace_bytes)(g.M, N, g.K);
    Tensor ws;
    if (ws_bytes) ws = make({ws_bytes}, at::kByte, out.device());
    void* wp = ws_bytes ? ws.data_ptr() : nullptr;
    const int bias_dtype = g.bias ? code(g.bias->scalar_type()) : LLMQ_BF16;
    if (g.fp8)
        check(llmq_gemm_fp8((const uint8_t*)g.q, LLMQ_E4M3, g.K, (const uint8_t*)g.w.data_ptr(), g.K, g.a_scale, g.w_scale, 1.f,
                            g.alpha, ptr(g.bias), bias_dtype, 1.f, out.data_ptr(), code(out_dtype), N, g.M, N, g.K, nullptr, wp,
                            (size_t)ws_bytes, l.stream),
              "llmq_gemm_fp8");
    else
        check(llmq_gemm_w8a8((const int8_t*)g.q, g.K, (const int8_t*)g.w.data_ptr(), g.K, g.a_scale, g.w_scale, 1.f, g.alpha,
                             ptr(g.bias), bias_dtype, 1.f, out.data_ptr(), code(out_dtype), N, g.M, N, g.K, nullptr, wp,
                             (size_t)ws_bytes, l.stream),
              "llmq_gemm_w8a8");
}

// ---- SmoothQuant int8 ------------------------------------------------------------------------------------------
// bias null: the output dtype is the activations' (the general path passes zeros of that dtype)
std::optional<Tensor> sq_tensor(const Tensor& x, const Tensor& w, const Tensor& w_scale, const std::optional<Tensor>& bias,
                                const Tensor& input_scale) {
    const Rows r = rows_of(x);
    if (!r.ok || !is16(x.scalar_type()) || !weight_ok(w, at::kChar, x.device(), r.K) || !scale_ok(w_scale, x.device(), 1) ||
        !bias_ok(bias, x.device(), w.size(0)) || (bias && !is16(bias->scalar_type())) || input_scale.device() != x.device())
        return std::nullopt;
    const at::ScalarType odt = bias ? bias->scalar_type() : x.scalar_type();
    const Launch l(x.device());
    if (one_launch(LLMQ_LINEAR_I8_TENSOR, r.M, w.size(0), r.K)) {
        Tensor out = make(out_size(x, w.size(0)), odt, x.device());
        check(llmq_linear_one_launch(LLMQ_LINEAR_I8_TENSOR, x.data_ptr(), code(x.scalar_type()), r.K, w.data_ptr(), r.K,
                                     (const float*)w_scale.data_ptr(), nullptr, ptr(bias), code(odt), nullptr, out.data_ptr(), code(odt),
                                     w.size(0), r.M, w.size(0), r.K, l.stream),
              "llmq_linear_one_launch");
        return out;
    }
    // codes, then {scale, alpha}, then the quantizer's partial maxima
    const int64_t codes = round16(r.M * r.K), part = (int64_t)llmq_quant_workspace_bytes();
    Tensor tmp = make({codes + 16 + part}, at::kByte, x.device());
    uint8_t* p = (uint8_t*)tmp.data_ptr();
    float* s = (float*)(p + codes);
    check(llmq_quant_per_tensor_alpha(0, x.data_ptr(), code(x.scalar_type()), r.M, r.K, r.K, p, s, (const float*)w_scale.data_ptr(),
                                      s + 1, p + codes + 16, (size_t)part, l.stream),
          "llmq_quant_per_tensor_alpha");
    Tensor out = make(out_size(x, w.size(0)), odt, x.device());
    gemm({false, p, w, nullptr, nullptr, s + 1, bias, r.M, r.K}, out, odt, l);
    return out;
}

std::optional<Tensor> sq_token(const Tensor& x, const Tensor& w, const Tensor& w_scale, const std::optional<Tensor>& bias) {
    const Rows r = rows_of(x);
    if (!r.ok || !is16(x.scalar_type()) || !weight_ok(w, at::kChar, x.device(), r.K)) return std::nullopt;
    const int64_t N = w.size(0);
    if (!scale_ok(w_scale, x.device(), N) || !bias_ok(bias, x.device(), N) || (bias && !is16(bias->scalar_type())))
        return std::nullopt;
    const at::ScalarType odt = bias ? bias->scalar_type() : x.scalar_type();
    const Launch l(x.device());
    const float* ws = (const float*)w_scale.data_ptr();
    Tensor out = make(out_size(x, N), odt, x.device());
    if (one_launch(LLMQ_LINEAR_I8_TOKEN, r.M, N, r.K)) {
        check(llmq_linear_one_launch(LLMQ_LINEAR_I8_TOKEN, x.data_ptr(), code(x.scalar_type()), r.K, w.data_ptr(), r.K, ws, nullptr, ptr(bias),
                                     code(odt), nullptr, out.data_ptr(), code(odt), N, r.M, N, r.K, l.stream),
              "llmq_linear_one_launch");
        return out;
    }
    const int64_t codes = round16(r.M * r.K);
    Tensor tmp = make({codes + 4 * r.M}, at::kByte, x.device());
    uint8_t* p = (uint8_t*)tmp.data_ptr();
    float* s = (float*)(p + codes);
    check(llmq_quant_i8_per_token(x.data_ptr(), code(x.scalar_type()), r.M, r.K, r.K, (int8_t*)p, s, LLMQ_F32, l.stream),
          "llmq_quant_i8_per_token");
    gemm({false, p, w, s, ws, nullptr, bias, r.M, r.K}, out, odt, l);
    return out;
}

// activations already quantized per token: codes [.., K] and fp32 scales, one per token
std::optional<Tensor> prequantized(bool fp8, const Tensor& q, const Tensor& a_scale, const Tensor& w, const Tensor& w_scale,
                                   const std::optional<Tensor>& bias, at::ScalarType odt) {
    const at::ScalarType qdt = fp8 ? at::kFloat8_e4m3fn : at::kChar;
    const Rows r = rows_of(q);
    if (!r.ok || q.scalar_type() != qdt || !weight_ok(w, qdt, q.device(), r.K)) return std::nullopt;
    const int64_t N = w.size(0);
    if (!scale_ok(a_scale, q.device(), r.M) || !scale_ok(w_scale, q.device(), N) || !bias_ok(bias, q.device(), N))
        return std::nullopt;
    if (bias && !(fp8 ? (bias->scalar_type() == at::kBFloat16 || bias->scalar_type() == at::kFloat) : is16(bias->scalar_type())))
        return std::nullopt;
    if (fp8) odt = at::kBFloat16;
    else if (bias) odt = bias->scalar_type();
    if (!is16(odt)) return std::nullopt;
    const Launch l(q.device());
    Tensor out = make(out_size(q, N), odt, q.device());
    gemm({fp8, q.data_ptr(), w, (const float*)a_scale.data_ptr(), (const float*)w_scale.data_ptr(), nullptr, bias, r.M, r.K}, out,
         odt, l);
    return out;
}

// ---- FP8 (e4m3fn) ----------------------------------------------------------------------------------------------
std::optional<Tensor> fp8_token(const Tensor& x, const Tensor& w, const Tensor& w_scale, const std::optional<Tensor>& bias) {
    const Rows r = rows_of(x);
    if (!r.ok || !is16(x.scalar_type()) || !weight_ok(w, at::kFloat8_e4m3fn, x.device(), r.K)) return std::nullopt;
    const int64_t N = w.size(0);
    if (!scale_ok(w_scale, x.device(), N) || !bias_ok(bias, x.device(), N) ||
        (bias && bias->scalar_type() != at::kBFloat16 && bias->scalar_type() != at::kFloat))
        return std::nullopt;
    const Launch l(x.device());
    const float* ws = (const float*)w_scale.data_ptr();
    Tensor out = make(out_size(x, N), at::kBFloat16, x.device());
    if (one_launch(LLMQ_LINEAR_FP8_TOKEN, r.M, N, r.K)) {
        check(llmq_linear_one_launch(LLMQ_LINEAR_FP8_TOKEN, x.data_ptr(), code(x.scalar_type()), r.K, w.data_ptr(), r.K, ws, nullptr, ptr(bias),
                                     bias ? code(bias->scalar_type()) : LLMQ_BF16, nullptr, out.data_ptr(), LLMQ_BF16, N, r.M, N, r.K,
                                     l.stream),
              "llmq_linear_one_launch");
        return out;
    }
    const int64_t codes = round16(r.M * r.K);
    Tensor tmp = make({codes + 4 * r.M}, at::kByte, x.device());
    uint8_t* p = (uint8_t*)tmp.data_ptr();
    float* s = (float*)(p + codes);
    check(llmq_quant_fp8_per_token(x.data_ptr(), code(x.scalar_type()), r.M, r.K, r.K, p, s, l.stream), "llmq_quant_fp8_per_token");
    gemm({true, p, w, s, ws, nullptr, bias, r.M, r.K}, out, at::kBFloat16, l);
    return out;
}

// Per-tensor scales.  input_scale absent: dynamic; present: static.  output_scale present: the result makes a round trip
// through e4m3fn on it and is fp32.
std::optional<Tensor> fp8_tensor(const Tensor& x, const Tensor& w, const Tensor& w_scale, const std::optional<Tensor>& bias,
                                 at::ScalarType odt, const std::optional<Tensor>& input_scale,
                                 const std::optional<Tensor>& output_scale) {
    const Rows r = rows_of(x);
    if (!r.ok || !is16(x.scalar_type()) || !is16(odt) || !weight_ok(w, at::kFloat8_e4m3fn, x.device(), r.K)) return std::nullopt;
    const int64_t N = w.size(0);
    if (!scale_ok(w_scale, x.device(), 1) || !bias_ok(bias, x.device(), N) || (bias && bias->scalar_type() != odt) ||
        (input_scale && (!scale_ok(*input_scale, x.device(), 1) || input_scale->dim() == 0)) ||
        (output_scale && !scale_ok(*output_scale, x.device(), 1)))
        return std::nullopt;
    const Launch l(x.device());
    const int kind = input_scale ? LLMQ_LINEAR_FP8_STATIC : LLMQ_LINEAR_FP8_TENSOR;
    if ((input_scale || !output_scale) && one_launch(kind, r.M, N, r.K)) {
        Tensor out = make(out_size(x, N), output_scale ? at::kFloat : odt, x.device());
        check(llmq_linear_one_launch(kind, x.data_ptr(), code(x.scalar_type()), r.K, w.data_ptr(), r.K, (const float*)w_scale.data_ptr(),
                                     input_scale ? (const float*)input_scale->data_ptr() : nullptr, ptr(bias), code(odt),
                                     output_scale ? (const float*)output_scale->data_ptr() : nullptr, out.data_ptr(), code(odt), N, r.M, N,
                                     r.K, l.stream),
              "llmq_linear_one_launch");
        return out;
    }
    const int64_t codes = round16(r.M * r.K), part = input_scale ? 0 : (int64_t)llmq_quant_workspace_bytes();
    Tensor tmp = make({codes + 16 + part}, at::kByte, x.device());
    uint8_t* p = (uint8_t*)tmp.data_ptr();
    float* s = (float*)(p + codes);
    const float* ws = (const float*)w_scale.data_ptr();
    if (input_scale)
        check(llmq_quant_fp8_static_alpha(x.data_ptr(), code(x.scalar_type()), r.M, r.K, r.K, p, (const float*)input_scale->data_ptr(),
                                          1, ws, s + 1, l.stream),
              "llmq_quant_fp8_static_alpha");
    else
        check(llmq_quant_per_tensor_alpha(1, x.data_ptr(), code(x.scalar_type()), r.M, r.K, r.K, p, s, ws, s + 1, p + codes + 16,
                                          (size_t)part, l.stream),
              "llmq_quant_per_tensor_alpha");
    if (!output_scale) {
        Tensor out = make(out_size(x, N), odt, x.device());
        gemm({true, p, w, nullptr, nullptr, s + 1, bias, r.M, r.K}, out, odt, l);
        return out;
    }
    Tensor out = make(out_size(x, N), at::kFloat, x.device());
    const int64_t ws_bytes = (int64_t)llmq_gemm_fp8_quantized_output_workspace_bytes(r.M, N, r.K);
    Tensor scratch;
    if (ws_bytes) scratch = make({ws_bytes}, at::kByte, x.device());
    check(llmq_gemm_fp8_quantized_output(p, LLMQ_E4M3, r.K, (const uint8_t*)w.data_ptr(), r.K, nullptr, nullptr, 1.f, s + 1, ptr(bias),
                                         code(odt), 1.f, (const float*)output_scale->data_ptr(), (float*)out.data_ptr(), code(odt),
                                         N, r.M, N, r.K, ws_bytes ? scratch.data_ptr() : nullptr, (size_t)ws_bytes, l.stream),
          "llmq_gemm_fp8_quantized_output");
    return out;
}

// ---- AWQ -------------------------------------------------------------------------------------------------------
// Arrival counters of the few-token kernel, one zeroed set per device and stream; every call leaves its set zero.
// A capture gets a set of its own per stream, zeroed by one node at its first use in the graph: the graph may be replayed on
// any stream, beside eager calls on the stream it was captured on, and after release().  That set is kept until the stream
// is next seen outside this capture; its memory is the graph's.  (Measured, four captured calls of a 7B layer at
// 1 / 4 tokens: 46.1 / 54.4 us; with a set and a fill node for each of the four 53.1 / 61.4.)
class CounterPool {
  public:
    static constexpr size_t kMaxStreams = 256;  // 128 MiB over all devices; streams past it pay for a zero fill per call
    Tensor get(const at::Device& dev, llmq_stream_t stream) {
        const bool capturing = c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
        unsigned long long id = 0;
        if (capturing) {
            hipStreamCaptureStatus status;
            if (hipStreamGetCaptureInfo((hipStream_t)stream, &status, &id) != hipSuccess) id = 0;
        }
        std::lock_guard<std::mutex> lock(mutex_);
        const Key key{dev.index(), stream};
        auto it = pool_.find(key);
        if (it == pool_.end()) {
            if (pool_.size() >= kMaxStreams || (capturing && id == 0)) return fresh(dev, stream);
            it = pool_.emplace(key, Sets{}).first;
        }
        Sets& s = it->second;
        if (capturing) {
            if (id == 0) return fresh(dev, stream);
            if (s.capture != id) s.captured = fresh(dev, stream), s.capture = id;
            return s.captured;
        }
        if (s.capture) s.captured.reset(), s.capture = 0;
        if (!s.eager.defined()) s.eager = fresh(dev, stream);
        return s.eager;
    }
    void release() {
        std::unordered_map<Key, Sets, Hash> old;
        std::lock_guard<std::mutex> lock(mutex_);
        old.swap(pool_);
    }

  private:
    struct Key {
        int dev;
        llmq_stream_t stream;
        bool operator==(const Key& o) const { return dev == o.dev && stream == o.stream; }
    };
    struct Hash {
        size_t operator()(const Key& k) const { return std::hash<void*>()(k.stream) * 31u + (size_t)k.dev; }
    };
    struct Sets {
        Tensor eager, captured;
        unsigned long long capture = 0;  // the capture that `captured` belongs to
    };
    static Tensor fresh(const at::Device& dev, llmq_stream_t stream) {
        const int64_t bytes = (int64_t)llmq_awq_workspace_ticket_bytes();
        Tensor t = make({bytes}, at::kByte, dev);
        check(llmq_awq_workspace_init(t.data_ptr(), (size_t)bytes, stream), "llmq_awq_workspace_init");
        return t;
    }
    std::mutex mutex_;
    std::unordered_map<Key, Sets, Hash> pool_;
};
CounterPool& counters() {
    static CounterPool* pool = new CounterPool;  // never destroyed: tensors must not outlive the allocator at exit
    return *pool;
}

// many_tokens: token count from which the weights are dequantized once and the fp16 GEMM runs
std::optional<Tensor> awq(const Tensor& x, const Tensor& qweight, const Tensor& qzeros, const Tensor& scales,
                          const std::optional<Tensor>& bias, int64_t group, int64_t many_tokens) {
    const Rows r = rows_of(x);
    if (!r.ok || !is16(x.scalar_type())) return std::nullopt;
    const at::Device dev = x.device();
    if (qweight.dim() != 2 || qweight.scalar_type() != at::kInt || qweight.size(0) != r.K || !plain_on(qweight, dev) || !aligned(qweight))
        return std::nullopt;
    const int64_t N = qweight.size(1) * 8;
    if (group <= 0 || r.K % group || group % 32 || (group != 32 && group != 64 && group != 128 && group != r.K)) return std::nullopt;
    if (qzeros.dim() != 2 || qzeros.scalar_type() != at::kInt || qzeros.size(0) != r.K / group || qzeros.size(1) * 8 != N ||
        !plain_on(qzeros, dev) || !aligned(qzeros) || scales.dim() != 2 || scales.scalar_type() != at::kHalf ||
        scales.size(0) != r.K / group || scales.size(1) != N || !plain_on(scales, dev) || !aligned(scales) ||
        !bias_ok(bias, dev, N) || (bias && bias->scalar_type() != at::kHalf) || N == 0)
        return std::nullopt;
    const Launch l(dev);
    const bool bf16 = x.scalar_type() == at::kBFloat16;
    if (r.M >= many_tokens) {
        const Tensor xh = bf16 ? x.to(at::kHalf) : x;
        Tensor w = make({N, r.K}, at::kHalf, dev);
        check(llmq_awq_dequant_t((const int32_t*)qweight.data_ptr(), scales.data_ptr(), (const int32_t*)qzeros.data_ptr(), w.data_ptr(),
                                 r.K, N, group, l.stream),
              "llmq_awq_dequant_t");
        Tensor out = make(out_size(x, N), at::kHalf, dev);
        const int64_t ws_bytes = (int64_t)llmq_gemm_f16_workspace_bytes(r.M, N, r.K);
        Tensor ws;
        if (ws_bytes) ws = make({ws_bytes}, at::kByte, dev);
        check(llmq_gemm_f16(xh.data_ptr(), r.K, w.data_ptr(), r.K, 1.f, ptr(bias), LLMQ_F16, 1.f, out.data_ptr(), LLMQ_F16, N, r.M, N,
                            r.K, nullptr, ws_bytes ? ws.data_ptr() : nullptr, (size_t)ws_bytes, l.stream),
              "llmq_gemm_f16");
        return bf16 ? out.to(at::kBFloat16) : out;
    }
    const bool native_bf16 = bf16 && llmq_awq_linear_bf16_supported(r.M, N, r.K, group, r.K);
    const Tensor xin = bf16 && !native_bf16 ? x.to(at::kHalf) : x;
    Tensor out = make(out_size(x, N), xin.scalar_type(), dev);
    // the partial sums of this call, and the arrival counters where the kernel that runs uses them
    const int xdt = native_bf16 ? LLMQ_BF16 : LLMQ_F16;
    int count = 0;
    const int64_t part = (int64_t)llmq_awq_linear_partials_bytes(xdt, r.M, N, r.K, group, r.K, &count);
    Tensor ws, tk;
    if (part) ws = make({part}, at::kByte, dev);
    if (count) tk = counters().get(dev, l.stream);
    check(llmq_awq_linear(xin.data_ptr(), xdt, r.K, (const int32_t*)qweight.data_ptr(), scales.data_ptr(), (const int32_t*)qzeros.data_ptr(),
                          ptr(bias), out.data_ptr(), r.M, N, r.K, group, count ? tk.data_ptr() : nullptr, part ? ws.data_ptr() : nullptr,
                          (size_t)part, l.stream),
          "llmq_awq_linear");
    return bf16 && !native_bf16 ? out.to(at::kBFloat16) : out;
}

// ---- RMSNorm ---------------------------------------------------------------------------------------------------
bool norm_ok(const Tensor& x, const Tensor& w, const Rows& r) {
    return r.ok && is16(x.scalar_type()) && r.K % 8 == 0 && w.defined() && w.scalar_type() == x.scalar_type() && w.numel() == r.K &&
           plain_on(w, x.device()) && aligned(w);
}
std::optional<Tensor> rmsnorm(const Tensor& x, const Tensor& w, double eps) {
    const Rows r = rows_of(x);
    if (!norm_ok(x, w, r)) return std::nullopt;
    const Launch l(x.device());
    Tensor y = make(x.sizes(), x.scalar_type(), x.device());
    check(llmq_rmsnorm(x.data_ptr(), code(x.scalar_type()), r.M, r.K, r.K, w.data_ptr(), (float)eps, y.data_ptr(), nullptr, l.stream),
          "llmq_rmsnorm");
    return y;
}
std::optional<std::pair<Tensor, Tensor>> rmsnorm_quant(const Tensor& x, const Tensor& w, double eps, bool fp8) {
    const Rows r = rows_of(x);
    if (!norm_ok(x, w, r)) return std::nullopt;
    const Launch l(x.device());
    Tensor q = make(x.sizes(), fp8 ? at::kFloat8_e4m3fn : at::kChar, x.device());
    Tensor s = make(out_size(x, 1), at::kFloat, x.device());
    if (fp8)
        check(llmq_rmsnorm_quant_fp8_per_token(x.data_ptr(), code(x.scalar_type()), r.M, r.K, r.K, w.data_ptr(), (float)eps, nullptr,
                                               (uint8_t*)q.data_ptr(), (float*)s.data_ptr(), nullptr, l.stream),
              "llmq_rmsnorm_quant_fp8_per_token");
    else
        check(llmq_rmsnorm_quant_i8_per_token(x.data_ptr(), code(x.scalar_type()), r.M, r.K, r.K, w.data_ptr(), (float)eps, nullptr,
                                              (int8_t*)q.data_ptr(), s.data_ptr(), LLMQ_F32, nullptr, l.stream),
              "llmq_rmsnorm_quant_i8_per_token");
    return std::make_pair(q, s);
}

// ---- Python ----------------------------------------------------------------------------------------------------
struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

// Positional arguments of a call: tensors by reference, None as an absent tensor.
struct Args {
    PyObject* const* a;
    bool all_tensors = true;
    const Tensor& tensor(int i) {
        static const Tensor none;
        if (!THPVariable_Check(a[i])) {
            all_tensors = false;
            return none;
        }
        return THPVariable_Unpack(a[i]);
    }
    std::optional<Tensor> optional(int i) {
        if (a[i] == Py_None) return std::nullopt;
        const Tensor& t = tensor(i);
        return all_tensors ? std::optional<Tensor>(t) : std::nullopt;
    }
    at::ScalarType dtype(int i) {
        if (!THPDtype_Check(a[i])) {
            all_tensors = false;
            return at::kFloat;
        }
        return reinterpret_cast<THPDtype*>(a[i])->scalar_type;
    }
};

PyObject* wrap(std::optional<Tensor>&& t) {
    if (!t) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(*t));
}
bool count_ok(Py_ssize_t n, Py_ssize_t want) {
    if (n == want) return true;
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
    return false;
}

#define LLMQ_PY(NAME, COUNT) PyObject* NAME(PyObject*, PyObject* const* argv, Py_ssize_t argc) { \
    HANDLE_TH_ERRORS                                                                             \
    if (!count_ok(argc, COUNT)) return nullptr;                                                  \
    Args in{argv};
#define LLMQ_PY_END  END_HANDLE_TH_ERRORS }
#define LLMQ_PY_TENSORS if (!in.all_tensors) Py_RETURN_NONE

LLMQ_PY(py_sq_tensor, 5)
    const Tensor &x = in.tensor(0), &w = in.tensor(1), &s = in.tensor(2), &is = in.tensor(4);
    const auto bias = in.optional(3);
    LLMQ_PY_TENSORS;
    std::optional<Tensor> y;
    { NoGil g; y = sq_tensor(x, w, s, bias, is); }
    return wrap(std::move(y));
LLMQ_PY_END

LLMQ_PY(py_sq_token, 4)
    const Tensor &x = in.tensor(0), &w = in.tensor(1), &s = in.tensor(2);
    const auto bias = in.optional(3);
    LLMQ_PY_TENSORS;
    std::optional<Tensor> y;
    { NoGil g; y = sq_token(x, w, s, bias); }
    return wrap(std::move(y));
LLMQ_PY_END

LLMQ_PY(py_sq_prequantized, 6)
    const Tensor &q = in.tensor(0), &a = in.tensor(1), &w = in.tensor(2), &s = in.tensor(3);
    const auto bias = in.optional(4);
    const at::ScalarType odt = in.dtype(5);
    LLMQ_PY_TENSORS;
    std::optional<Tensor> y;
    { NoGil g; y = prequantized(false, q, a, w, s, bias, odt); }
    return wrap(std::move(y));
LLMQ_PY_END

LLMQ_PY(py_fp8_prequantized, 5)
    const Tensor &q = in.tensor(0), &a = in.tensor(1), &w = in.tensor(2), &s = in.tensor(3);
    const auto bias = in.optional(4);
    LLMQ_PY_TENSORS;
    std::optional<Tensor> y;
    { NoGil g; y = prequantized(true, q, a, w, s, bias, at::kBFloat16); }
    return wrap(std::move(y));
LLMQ_PY_END

LLMQ_PY(py_fp8_token, 4)
    const Tensor &x = in.tensor(0), &w = in.tensor(1), &s = in.tensor(2);
    const auto bias = in.optional(3);
    LLMQ_PY_TENSORS;
    std::optional<Tensor> y;
    { NoGil g; y = fp8_token(x, w, s, bias); }
    return wrap(std::move(y));
LLMQ_PY_END

LLMQ_PY(py_fp8_tensor, 7)
    const Tensor &x = in.tensor(0), &w = in.tensor(1), &s = in.tensor(2);
    const auto bias = in.optional(3);
    const at::ScalarType odt = in.dtype(4);
    const auto input_scale = in.optional(5), output_scale = in.optional(6);
    LLMQ_PY_TENSORS;
    std::optional<Tensor> y;
    { NoGil g; y = fp8_tensor(x, w, s, bias, odt, input_scale, output_scale); }
    return wrap(std::move(y));
LLMQ_PY_END

LLMQ_PY(py_awq, 7)
    const Tensor &x = in.tensor(0), &qw = in.tensor(1), &qz = in.tensor(2), &s = in.tensor(3);
    const auto bias = in.optional(4);
    LLMQ_PY_TENSORS;
    const long long group = PyLong_AsLongLong(argv[5]), many = PyLong_AsLongLong(argv[6]);
    if (PyErr_Occurred()) return nullptr;
    std::optional<Tensor> y;
    { NoGil g; y = awq(x, qw, qz, s, bias, group, many); }
    return wrap(std::move(y));
LLMQ_PY_END

LLMQ_PY(py_rmsnorm, 3)
    const Tensor &x = in.tensor(0), &w = in.tensor(1);
    LLMQ_PY_TENSORS;
    const double eps = PyFloat_AsDouble(argv[2]);
    if (PyErr_Occurred()) return nullptr;
    std::optional<Tensor> y;
    { NoGil g; y = rmsnorm(x, w, eps); }
    return wrap(std::move(y));
LLMQ_PY_END

LLMQ_PY(py_rmsnorm_quant, 4)
    const Tensor &x = in.tensor(0), &w = in.tensor(1);
    LLMQ_PY_TENSORS;
    const double eps = PyFloat_AsDouble(argv[2]);
    const int fp8 = PyObject_IsTrue(argv[3]);
    if (PyErr_Occurred()) return nullptr;
    std::optional<std::pair<Tensor, Tensor>> y;
    { NoGil g; y = rmsnorm_quant(x, w, eps, fp8 != 0); }
    if (!y) Py_RETURN_NONE;
    PyObject* q = THPVariable_Wrap(std::move(y->first));
    PyObject* s = q ? THPVariable_Wrap(std::move(y->second)) : nullptr;
    PyObject* both = s ? PyTuple_Pack(2, q, s) : nullptr;
    Py_XDECREF(q);
    Py_XDECREF(s);
    return both;
LLMQ_PY_END

// the counters of the current stream of a tensor's device
LLMQ_PY(py_awq_counters, 1)
    const Tensor& x = in.tensor(0);
    LLMQ_PY_TENSORS;
    if (!x.is_cuda()) Py_RETURN_NONE;
    Tensor t;
    {
        NoGil g;
        const Launch l(x.device());
        t = counters().get(x.device(), l.stream);
    }
    return THPVariable_Wrap(std::move(t));
LLMQ_PY_END

PyObject* py_release_counters(PyObject*, PyObject*) {
    HANDLE_TH_ERRORS
    {
        NoGil g;  // a thread inside get() may wait for the interpreter lock (allocator hooks)
        counters().release();
    }
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

#define LLMQ_FAST(NAME, FN) {NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(FN)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {LLMQ_FAST("sq_tensor", py_sq_tensor),
                         LLMQ_FAST("sq_token", py_sq_token),
                         LLMQ_FAST("sq_prequantized", py_sq_prequantized),
                         LLMQ_FAST("fp8_prequantized", py_fp8_prequantized),
                         LLMQ_FAST("fp8_token", py_fp8_token),
                         LLMQ_FAST("fp8_tensor", py_fp8_tensor),
                         LLMQ_FAST("awq", py_awq),
                         LLMQ_FAST("rmsnorm", py_rmsnorm),
                         LLMQ_FAST("rmsnorm_quant", py_rmsnorm_quant),
                         LLMQ_FAST("awq_counters", py_awq_counters),
                         {"release_tickets", py_release_counters, METH_NOARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_llmq_host", "native forward passes of the quantized modules", -1, methods,
                          nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" PyObject* PyInit__llmq_host(void) {
    PyObject* m = PyModule_Create(&module_def);
    // the tensors that cross this boundary have the layout of the torch it was compiled against
    if (m && PyModule_AddStringConstant(m, "torch_version", LLMQ_TORCH_VERSION) != 0) Py_CLEAR(m);
    return m;
}
