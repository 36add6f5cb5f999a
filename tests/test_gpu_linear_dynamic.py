"""GPU parity of the one-launch few-token linears (per-token dynamic quantizer + GEMM + epilogue):
codes, scales and raw accumulators against the oracle, outputs bit-identical to the two-launch form."""
import pytest
import torch

from oracle import ref_math as R

pytestmark = pytest.mark.gpu

# (K, N): Qwen2-7B qkv and down, a ragged channel edge with an odd number of K steps plus a 16-byte tail, one step
SHAPES = [(3584, 4608), (18944, 3584), (1040, 264), (64, 40)]


@pytest.fixture
def force_variant():
    from llmqrt_amd import _abi
    yield lambda v: _abi.check(_abi.lib().llmq_linear_dynamic_force_variant(v), "force_variant")
    _abi.lib().llmq_linear_dynamic_force_variant(-1)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 3, 16])
@pytest.mark.parametrize("K,N", SHAPES)
def test_int8_dynamic_linear(cuda, force_variant, variant, dtype, M, K, N):
    from llmqrt_amd import workloads as W
    from llmqrt_amd.sq_fp8_kernels import dynamic_linear_max_tokens
    if M > dynamic_linear_max_tokens(K):
        pytest.skip("the quantized rows of this many tokens do not fit in LDS at this K")
    from llmqrt_amd.quantize import quantize_activation_per_token_absmax_f32
    from llmqrt_amd.sq_fp8_kernels import w8a8_int8_linear_bbf16_obf16_per_channel, w8a8_int8_linear_dynamic_per_token
    x = W.activations(M, 2 * K, 900 + M + K, dtype=dtype)[:, :K]   # row stride 2K
    qw, sw = W.int8_weights(N, K, 901 + N)
    bias = (0.1 * torch.randn(N, generator=torch.Generator().manual_seed(N))).to(dtype)
    q_ref, s_ref = R.quantize_activation_per_token_absmax(x)
    acc_ref = R.int8_gemm_exact(q_ref, qw)
    xd = W.activations(M, 2 * K, 900 + M + K, dtype=dtype).to(cuda)[:, :K]
    assert xd.stride(0) == 2 * K
    args = (qw.to(cuda).t(), bias.to(cuda), sw.to(cuda))
    force_variant(variant)
    qd = torch.full((M, K), 99, dtype=torch.int8, device=cuda)
    sd = torch.zeros(M, dtype=torch.float32, device=cuda)
    ad = torch.full((M, N), -5, dtype=torch.int32, device=cuda)
    y = w8a8_int8_linear_dynamic_per_token(xd, *args, _q_dump=qd, _scale_dump=sd, _acc_dump=ad)
    assert y.dtype == dtype and y.shape == (M, N)
    assert torch.equal(qd.cpu(), q_ref), "codes"
    assert torch.equal(sd.cpu(), s_ref.float().view(-1)), "scales"
    assert torch.equal(ad.cpu(), acc_ref), "int32 accumulators"
    q2, s2 = quantize_activation_per_token_absmax_f32(xd.contiguous())
    two = w8a8_int8_linear_bbf16_obf16_per_channel(q2, args[0], args[1], s2, args[2])
    assert torch.equal(y.view(torch.int16), two.view(torch.int16)), "same bits as quantizer + GEMM"
    assert torch.equal(y, w8a8_int8_linear_dynamic_per_token(xd, *args)), "deterministic, dumps optional"


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 3, 16])
@pytest.mark.parametrize("K,N", SHAPES)
def test_fp8_dynamic_linear(cuda, force_variant, variant, dtype, M, K, N):
    from llmqrt_amd import _abi, workloads as W
    from llmqrt_amd.sq_fp8_kernels import dynamic_linear_max_tokens
    if M > dynamic_linear_max_tokens(K):
        pytest.skip("the quantized rows of this many tokens do not fit in LDS at this K")
    from llmqrt_amd.quantize import per_token_quantize
    from llmqrt_amd.sq_fp8_kernels import cutlass_f8f8bf16_rowwise_sm89, f8f8bf16_linear_dynamic_per_token
    x = W.activations(M, K, 910 + M + K, dtype=dtype)
    wq, ws = W.fp8_weights(N, K, 911 + N)
    bias = (0.1 * torch.randn(N, generator=torch.Generator().manual_seed(N))).bfloat16()
    q_ref, s_ref = R.fp8_per_token_quantize(x)
    xd = x.to(cuda)
    wsd = ws.to(cuda).float().reshape(-1).contiguous()
    force_variant(variant)
    qd = torch.zeros((M, K), dtype=torch.uint8, device=cuda)
    sd = torch.zeros(M, dtype=torch.float32, device=cuda)
    ad = torch.zeros((M, N), dtype=torch.float32, device=cuda)
    y = f8f8bf16_linear_dynamic_per_token(xd, wq.to(cuda).t(), bias.to(cuda), wsd, _q_dump=qd, _scale_dump=sd, _acc_dump=ad)
    assert y.dtype == torch.bfloat16 and y.shape == (M, N)
    assert torch.equal(qd.cpu(), q_ref.view(torch.uint8)), "codes"
    assert torch.equal(sd.cpu(), s_ref.view(-1)), "scales"
    q2, s2 = per_token_quantize(xd)
    ad2 = torch.zeros((M, N), dtype=torch.float32, device=cuda)
    # the few-token GEMM with the same channel tiles per wavefront and wavefronts along K adds in the same order
    _abi.check(_abi.lib().llmq_gemm_force_plan(101 if variant == 0 else 102, 1), "force_plan")
    try:
        two = cutlass_f8f8bf16_rowwise_sm89(q2, wq.to(cuda).t(), bias.to(cuda), s2.view(-1, 1), wsd.view(1, -1), True, _acc_dump=ad2)
    finally:
        _abi.lib().llmq_gemm_force_plan(-1, 1)
    assert torch.equal(ad, ad2), "same fp32 accumulators as the few-token GEMM"
    assert torch.equal(y.view(torch.int16), two.view(torch.int16)), "same bits as quantizer + GEMM"
    y_ref = R.fp8_linear_naive(q_ref, s_ref, wq, ws, bias)
    assert ((y.float().cpu() - y_ref.float()).abs().max() / y_ref.float().abs().max()).item() <= 1e-2


def test_dynamic_linear_rejects_more_tokens_and_bad_layout(cuda):
    from llmqrt_amd import workloads as W
    from llmqrt_amd.sq_fp8_kernels import dynamic_linear_max_tokens, w8a8_int8_linear_dynamic_per_token
    mt = dynamic_linear_max_tokens(128)
    assert mt == 16 and dynamic_linear_max_tokens(18944) == 3 and dynamic_linear_max_tokens(3584) == 16
    qw, sw = W.int8_weights(64, 128, 5)
    bias = torch.zeros(64, dtype=torch.bfloat16, device=cuda)
    x = torch.zeros((mt + 1, 128), dtype=torch.bfloat16, device=cuda)
    with pytest.raises(RuntimeError):
        w8a8_int8_linear_dynamic_per_token(x, qw.to(cuda).t(), bias, sw.to(cuda))
    with pytest.raises(RuntimeError):
        w8a8_int8_linear_dynamic_per_token(x[:2].float(), qw.to(cuda).t(), bias, sw.to(cuda))
    empty = w8a8_int8_linear_dynamic_per_token(x[:0], qw.to(cuda).t(), bias, sw.to(cuda))
    assert empty.shape == (0, 64)


@pytest.mark.parametrize("tokens", [1, 4, 5])
def test_modules_take_the_one_launch_path_with_identical_results(cuda, tokens):
    """SqW8A8BBF16OBF16PerChannel and FP8DynamicLinear (per token) run these tokens in one launch and 17 in two:
    the result must not depend on which side of the switch a batch falls (rows of a 17-token batch = the same rows
    computed alone)."""
    from llmqrt_amd.linear import FP8DynamicLinear, SqW8A8BBF16OBF16PerChannel
    torch.manual_seed(3)
    dense = torch.nn.Linear(512, 384, bias=True).to(cuda)
    x = torch.randn(17, 512, device=cuda).to(torch.bfloat16)
    sq = SqW8A8BBF16OBF16PerChannel.from_linear(dense, 8, 0, init_only=False, dtype=torch.bfloat16)
    f8 = FP8DynamicLinear.from_linear(dense, init_only=False, dtype=torch.bfloat16, per_tensor=False)
    full, part = sq(x), sq(x[:tokens])    # 17 tokens: quantizer + GEMM; up to 5: one launch
    assert torch.equal(part, full[:tokens])   # int32 accumulation is exact, the epilogue arithmetic is shared
    full, part = f8(x), f8(x[:tokens])    # fp32 accumulation: the two kernels add in different orders
    assert ((part.float() - full[:tokens].float()).abs().max() / full.float().abs().max()).item() <= 1e-2


# One launch with a tensor-wide scale, native, against quantizer + GEMM, the general path of contiguous rows: one token, several, rows past the MFMA's 16-byte
# steps, one channel tile / two / ragged N; 2 x 4104 x 8192 takes two launches either way.  int8: the same bits as quantizer + GEMM; fp8: fp32
# sums of the same products, in another order where the GEMM is the tile kernel, then one rounding: a bf16 step is 2^-8.
@pytest.mark.parametrize("M,N,K", [(1, 3584, 3584), (4, 3584, 3584), (5, 3584, 3584), (16, 896, 896), (16, 1000, 1024), (2, 4104, 8192),
                                   (1, 520, 16384), (3, 9728, 912), (1, 5000, 2064), (16, 24, 16)])
@pytest.mark.parametrize("dtype,bias", [(torch.bfloat16, True), (torch.float16, False)])
def test_per_tensor_one_launch(cuda, M, N, K, dtype, bias):
    from llmqrt_amd.linear import FP8DynamicLinear, SqW8A8BBF16OBF16PerTensor
    g = torch.Generator(device="cuda").manual_seed(M + K)
    lin = torch.nn.Linear(K, N, bias=bias, device="cuda")
    lin.weight.data = 0.02 * torch.randn(N, K, device="cuda", generator=g)
    x = torch.randn(M, K, device="cuda", generator=g).to(dtype)
    x[-1, -1] = 50.0  # the largest value in the last piece of the last row
    sq = SqW8A8BBF16OBF16PerTensor.from_linear(lin, 8, 0, False, dtype=dtype)
    f8 = FP8DynamicLinear.from_linear(lin, init_only=False, dtype=dtype, per_tensor=True)
    for v in (x, torch.zeros_like(x)):
        assert torch.equal(sq(v), sq._forward_general(v))
        y, ref = f8(v).double(), f8._forward_general(v).double()
        assert torch.equal(y.isnan(), ref.isnan())  # fp16 zeros: the quantizer's floor is 0 in fp16, and 0 / 0 is NaN either way
        y, ref = y.nan_to_num(), ref.nan_to_num()
        assert (y - ref).abs().max() <= 2.0 ** -8 * ref.abs().max()
    x[0, 3] = float("nan")
    assert torch.equal(f8(x).isnan(), f8._forward_general(x).isnan())


# llmq_linear_one_launch in every launch shape: up to 4096 channels 2, 4 and 10 pieces a thread (the last and the first number of codes of each),
# past that four and eight wavefronts, one row per wavefront and several; a ragged K step, ragged channels, one step, LDS past 64 KB and codes of 64 KB exactly
@pytest.mark.parametrize("M,N,K", [(1, 24, 16), (16, 4096, 1024), (15, 1000, 1104), (16, 264, 2048), (16, 136, 2064), (16, 896, 4864), (16, 72, 5120), (16, 40, 4080), (8, 40, 8176), (1, 640, 16384),
                                   (4, 512, 20480), (8, 4112, 1024), (9, 4104, 1040), (16, 4360, 1024), (13, 8200, 1280), (3, 9728, 912), (16, 4112, 2064)])
@pytest.mark.parametrize("dtype,with_bias", [(torch.bfloat16, True), (torch.float16, False)])
def test_one_launch_every_source(cuda, M, N, K, dtype, with_bias):
    """Against quantizer + GEMM on the same operands: int8 bit for bit (exact int32 sums), fp8 within the rounding of two fp32 sums of the same
    products in different orders, K 2^-24 of the sum of their absolute values, and one rounding to the output type (or one step of e4m3fn)."""
    from llmqrt_amd import _abi, workloads as W
    from llmqrt_amd.quantize import per_token_quantize, quantize_activation_per_token_absmax_f32, static_per_tensor_quantize_with_alpha
    from llmqrt_amd.quantize import per_tensor_quantize_with_alpha
    from llmqrt_amd.sq_fp8_kernels import w8a8_int8_linear_bbf16_obf16_per_channel, w8a8_int8_linear_bbf16_obf16_per_tensor
    L = _abi.lib()
    g = torch.Generator().manual_seed(M + N + K)
    x = (torch.randn(M, K, generator=g) * 2).to(dtype).to(cuda)
    x[-1, -1] = 40.0
    qi, swi = (t.to(cuda) for t in W.int8_weights(N, K, N + 1))
    qf = (torch.randn(N, K, generator=g) * 60).clamp(-448, 448).to(torch.float8_e4m3fn).to(cuda)
    swn = (torch.rand(N, generator=g) * 0.01 + 0.001).to(cuda)
    sw1 = torch.tensor([0.004], device=cuda)
    sin = torch.tensor([0.0137], device=cuda)
    sout = torch.tensor([0.9], device=cuda)
    bias = torch.randn(N, generator=g).to(dtype).to(cuda) if with_bias else None
    bd = bias.double() if with_bias else 0

    def run(kind, w, sw, in_scale=None, out_scale=None):
        out = torch.full((M, N), 7.0, dtype=torch.float32 if out_scale is not None else dtype, device=cuda)
        _abi.check(L.llmq_linear_one_launch(kind, x.data_ptr(), _abi.dtype_code(dtype), K, w.data_ptr(), K, sw.data_ptr(), _abi.ptr(in_scale),
                                            _abi.ptr(bias), _abi.dtype_code(dtype), _abi.ptr(out_scale), out.data_ptr(), _abi.dtype_code(dtype), N,
                                            M, N, K, torch.cuda.current_stream().cuda_stream), "llmq_linear_one_launch")
        return out
    zeros = torch.zeros(N, dtype=dtype, device=cuda)
    b = bias if with_bias else zeros
    # int8
    q, s = quantize_activation_per_token_absmax_f32(x)
    assert torch.equal(run(0, qi, swn), w8a8_int8_linear_bbf16_obf16_per_channel(q, qi.t(), b, s, swn))
    q, alpha = per_tensor_quantize_with_alpha(x, sw1, fp8=False)
    assert torch.equal(run(2, qi, sw1), w8a8_int8_linear_bbf16_obf16_per_tensor(q.view(M, K), qi.t(), b, alpha, 1.0))
    # fp8: codes and scales of the separate quantizers, fp64 sums
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11

    def check(y, codes, scale, w_scale):
        prod = codes.double() @ qf.double().t() * scale.double() * w_scale.double()
        mag = codes.double().abs() @ qf.double().abs().t() * scale.double() * w_scale.double()
        ref = prod + bd
        # the matrix cores drop products more than 13 binary orders below the largest of a run of eight
        tol = (K * 2.0 ** -24 + 2.0 ** -13) * mag + 2.0 * ulp * ref.abs() + 2.0 ** -20
        assert bool(((y.double() - ref).abs() <= tol).all()), float(((y.double() - ref).abs() / tol).max())
        return ref, tol
    q, s = per_token_quantize(x)
    check(run(1, qf, swn), q.float(), s.view(M, 1), swn.view(1, N))
    q, alpha = per_tensor_quantize_with_alpha(x, sw1, fp8=True)
    check(run(3, qf, sw1), q.view(M, K).float(), alpha.view(1, 1), torch.ones(1, device=cuda))
    q, alpha = static_per_tensor_quantize_with_alpha(x, sin, sw1)
    ref, tol = check(run(4, qf, sw1, sin), q.view(M, K).float(), alpha.view(1, 1), torch.ones(1, device=cuda))
    y = run(4, qf, sw1, sin, sout)
    codes = y / sout
    assert torch.equal(codes.to(torch.float8_e4m3fn).float() * sout, y)  # on the grid
    step = (ref / 0.9).abs().clamp(min=2.0 ** -6, max=448.0)
    assert bool(((y.double() - ref.clamp(-448 * 0.9, 448 * 0.9)).abs() <= 0.9 * step * 2.0 ** -3 + tol).all())


def test_one_launch_refuses(cuda):
    from llmqrt_amd import _abi
    L = _abi.lib()
    x = torch.zeros(17, 8192, dtype=torch.bfloat16, device=cuda)
    w = torch.zeros(64, 8192, dtype=torch.int8, device=cuda)
    s = torch.ones(64, device=cuda)
    out = torch.zeros(17, 64, dtype=torch.bfloat16, device=cuda)

    def rc(kind, M, K, sw=s, sin=None, sout=None):
        return L.llmq_linear_one_launch(kind, x.data_ptr(), _abi.BF16, K, w.data_ptr(), K, _abi.ptr(sw), _abi.ptr(sin), None, 0, _abi.ptr(sout), out.data_ptr(),
                                        _abi.BF16, 64, M, 64, K, 0)
    assert rc(2, 17, 64) == rc(2, 11, 8192) == rc(5, 1, 64) == rc(-1, 1, 64) == rc(2, 1, 40) == -3  # LLMQ_ERR_SHAPE
    assert rc(2, 1, 64, None) == rc(4, 1, 64, s, None) == L.llmq_linear_one_launch(0, None, 0, 64, None, 64, None, None, None, 0, None, None, 0, 64, 1, 64, 64, 0)
    assert rc(2, 1, 64, None) != 0 and rc(3, 1, 64, s, None, s) != 0
    assert rc(2, 0, 64) == 0 and int(out.count_nonzero()) == 0
    for kind in range(5):
        assert L.llmq_linear_one_launch_preferred(kind, 17, 64, 64) == 0 == L.llmq_linear_one_launch_preferred(kind, 1, 64, 40)


def _modules(N, K, dtype, bias, cuda):
    from llmqrt_amd.linear import FP8DynamicLinear, FP8StaticLinear, SqW8A8BBF16OBF16PerChannel, SqW8A8BBF16OBF16PerTensor
    g = torch.Generator(device="cuda").manual_seed(N + K)
    lin = torch.nn.Linear(K, N, bias=bias, device="cuda")
    lin.weight.data = 0.02 * torch.randn(N, K, device="cuda", generator=g)
    if bias:
        lin.bias.data = torch.randn(N, device="cuda", generator=g)
    mods = {"sq": SqW8A8BBF16OBF16PerTensor.from_linear(lin, 8, 0, False, dtype=dtype),
            "sq_channel": SqW8A8BBF16OBF16PerChannel.from_linear(lin, 8, 0, False, dtype=dtype),
            "fp8": FP8DynamicLinear.from_linear(lin, init_only=False, dtype=dtype)}
    if dtype == torch.bfloat16:
        mods["fp8_token"] = FP8DynamicLinear.from_linear(lin, init_only=False, dtype=dtype, per_tensor=False)
    for name, quantized in (("static", False), ("static_out", True)):
        m = mods[name] = FP8StaticLinear.from_linear(lin, init_only=False, dtype=dtype, quantize_output=quantized)
        m.input_scale.data.fill_(0.03)
        m.output_scale.data.fill_(0.05)
    return mods


# one launch and two by every rule: few and many codes, up to 4096 channels and past them, more than 4 tokens, a ragged K, a K past 8192
@pytest.mark.parametrize("M,N,K", [(3, 896, 3584), (10, 3072, 3008), (16, 896, 4864), (8, 3584, 3584), (16, 9728, 896), (4, 20488, 1040), (2, 520, 12288), (13, 512, 2064)])
@pytest.mark.parametrize("dtype,bias", [(torch.bfloat16, True), (torch.float16, False)])
def test_strided_rows_give_the_bits_of_contiguous_ones(cuda, M, N, K, dtype, bias):
    """The same values in rows that are further apart (and start 16 bytes into the buffer) run the same kernels as contiguous ones, eager and captured."""
    wide = torch.zeros(M, 1, K + 24, dtype=dtype, device=cuda)
    wide[..., 8:8 + K] = (torch.randn(M, 1, K, device=cuda, generator=torch.Generator(device="cuda").manual_seed(M)) * 2).to(dtype)
    strided = wide[..., 8:8 + K]
    x = strided.contiguous()
    for name, mod in _modules(N, K, dtype, bias, cuda).items():
        want = mod(x)
        got = mod(strided)
        assert got.dtype == want.dtype and got.shape == want.shape and torch.equal(got, want), name
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            a, b = mod(x), mod(strided)
        for _ in range(2):
            graph.replay()
            mod(strided)
            torch.cuda.synchronize()
            assert torch.equal(a, b), name


@pytest.mark.parametrize("M,N,K", [(3, 896, 3584), (10, 3072, 3008), (16, 896, 4864), (16, 9728, 896), (4, 37504, 1408)])
def test_strided_rows_take_the_launch_of_contiguous_ones(cuda, M, N, K):
    """Where the rule says one launch a strided call makes its output and nothing else; where it says two (the per-token kinds of the last size), codes and
    scales as well."""
    from llmqrt_amd import _abi
    kinds = {"sq_channel": 0, "fp8_token": 1, "sq": 2, "fp8": 3, "static": 4, "static_out": 4}
    strided = torch.randn(M, K + 24, device=cuda, generator=torch.Generator(device="cuda").manual_seed(M)).bfloat16()[:, 8:8 + K]
    for name, mod in _modules(N, K, torch.bfloat16, True, cuda).items():
        mod(strided)
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        mod(strided)
        made = torch.cuda.memory_stats()["allocation.all.allocated"] - before
        one = _abi.lib().llmq_linear_one_launch_preferred(kinds[name], M, N, K)
        assert (made == 1) == bool(one), (name, made)


def test_strided_rows_off_the_kernel_still_run(cuda):
    """Rows, columns and addresses that no one-launch kernel takes: the general path copies or quantizes separately, as for any size."""
    M, N, K = 5, 640, 1024
    g = torch.Generator(device="cuda").manual_seed(1)
    wide = torch.randn(M, 2 * K + 13, device=cuda, generator=g).bfloat16()
    views = {"odd address": wide[:, 1:1 + K], "odd stride": wide[:, :K], "every other column": wide[:, :2 * K:2],
             "transposed": torch.randn(K, M, device=cuda, generator=g).bfloat16().t()}
    for name, mod in _modules(N, K, torch.bfloat16, True, cuda).items():
        for what, x in views.items():
            y, ref = mod(x).double(), mod(x.contiguous().clone()).double()
            assert y.shape == (M, N) and (y - ref).abs().max() <= 2.0 ** -7 * ref.abs().max() + (0.05 * 2.0 ** -3 if name == "static_out" else 0), (name, what)


@pytest.mark.parametrize("fp8", [0, 1])
@pytest.mark.parametrize("M,N,K", [(1, 24, 16), (16, 896, 1024), (4, 4104, 4096), (5, 9728, 912)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_per_tensor_entry_point(cuda, fp8, M, N, K, dtype):
    """llmq_linear_per_tensor_dynamic is llmq_linear_one_launch for up to llmq_linear_per_tensor_max_tokens tokens, and refuses more."""
    from llmqrt_amd import _abi
    L = _abi.lib()
    g = torch.Generator().manual_seed(N)
    x = torch.randn(M, K + 8, generator=g).to(dtype).to(cuda)
    w = (torch.randn(N, K, generator=g) * 40).clamp(-127, 127)
    w = (w.to(torch.float8_e4m3fn) if fp8 else w.to(torch.int8)).to(cuda)
    s = torch.tensor([0.01], device=cuda)
    bias = torch.randn(N, generator=g).to(dtype).to(cuda)
    a, b = (torch.zeros(M, N, dtype=dtype, device=cuda) for _ in range(2))
    dt, st = _abi.dtype_code(dtype), torch.cuda.current_stream().cuda_stream

    def entry(tokens):
        return L.llmq_linear_per_tensor_dynamic(fp8, x.data_ptr(), dt, K + 8, w.data_ptr(), K, s.data_ptr(), bias.data_ptr(), dt, a.data_ptr(), dt, N, tokens, N, K, st)
    assert entry(M) == 0 and entry(L.llmq_linear_per_tensor_max_tokens(K) + 1) == -3
    assert L.llmq_linear_one_launch(2 + fp8, x.data_ptr(), dt, K + 8, w.data_ptr(), K, s.data_ptr(), None, bias.data_ptr(), dt, None, b.data_ptr(), dt, N, M, N, K, st) == 0
    assert torch.equal(a, b) and int(a.count_nonzero()) > 0
