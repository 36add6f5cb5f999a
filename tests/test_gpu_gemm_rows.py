"""The few-token GEMM that streams long pieces of rows through LDS: every variant, at the sizes where it can go wrong."""
import pytest
import torch

from oracle import ref_math as R

pytestmark = pytest.mark.gpu

TOKENS = [16, 16, 16, 32, 32, 32, 32, 32, 48, 48, 64, 64, 16, 16]  # what a block of each variant holds


def _ints(shape, seed):
    return torch.randint(-127, 128, shape, generator=torch.Generator().manual_seed(seed), dtype=torch.int32).to(torch.int8)


# fewer tokens than a block holds, one, all; channels that end inside a 16-channel tile, inside a store of four, inside a block; K of one MFMA
# step's part, a stage, a stage and 16 bytes, more and fewer stages than LDS slots, a ragged end in the last of several
@pytest.mark.parametrize("variant", range(14))
@pytest.mark.parametrize("missing,N,K", [(0, 136, 16), (15, 37, 1024), (3, 72, 528), (0, 200, 2560), (1, 264, 3600), (5, 64, 7168), (0, 48, 9232)])
def test_every_variant(cuda, variant, missing, N, K):
    """Rows further apart than K, an output inside a larger one.  int8: accumulators and results bit for bit.  fp8 (e4m3 and e5m2
    activations): products are exact, so only the fp32 sums round: 2e-4 of the largest for what the matrix cores' accumulation window loses,
    and half a bf16 step; the quantized output is the three steps on that result bit for bit."""
    from llmqrt_amd import _abi
    from llmqrt_amd.quantize import static_per_tensor_quantize
    L = _abi.lib()
    M = max(1, TOKENS[variant] - missing)
    ld, ldo = K + 48, N + 5
    g = torch.Generator().manual_seed(N)
    sx, sw = torch.rand(M, generator=g) * 0.01 + 1e-3, torch.rand(N, generator=g) * 0.01 + 1e-3
    bias = torch.randn(N, generator=g).bfloat16()
    qx, qw = _ints((M, ld), M), _ints((N, ld), N + 1)
    a, b = [(torch.randn(n, ld, generator=g) * 30).clamp(-448, 448).to(torch.float8_e4m3fn) for n in (M, N)]
    a5 = a.float().to(torch.float8_e5m2)
    dev = [t.to(cuda) for t in (sx, sw, bias, qx, qw, a, b, a5)]
    p = [t.data_ptr() for t in dev]
    out = torch.full((M, ldo), 7.0, dtype=torch.bfloat16, device=cuda)
    dump = torch.full((M, N), -1, dtype=torch.int32, device=cuda)
    stream = torch.cuda.current_stream().cuda_stream
    _abi.check(L.llmq_gemm_force_plan(110 + variant, 1), "force_plan")
    try:
        _abi.check(L.llmq_gemm_w8a8(p[3], ld, p[4], ld, p[0], p[1], 1.0, None, p[2], 0, 1.0, out.data_ptr(), 0, ldo, M, N, K, dump.data_ptr(), None, 0, stream), "int8")
        y, f8 = out.clone(), []
        for fmt, x in ((0, p[5]), (1, p[7])):
            _abi.check(L.llmq_gemm_fp8(x, fmt, ld, p[6], ld, p[0], p[1], 1.0, None, p[2], 0, 1.0, out.data_ptr(), 0, ldo, M, N, K, None, None, 0, stream), "fp8")
            f8.append(out.clone())
        scale = f8[0][:, :N].float().abs().max() / 300
        quant = torch.full((M, ldo), 7.0, device=cuda)
        _abi.check(L.llmq_gemm_fp8_quantized_output(p[5], 0, ld, p[6], ld, p[0], p[1], 1.0, None, p[2], 0, 1.0, scale.data_ptr(), quant.data_ptr(), 0, ldo, M, N, K,
                                                    None, 0, stream), "fp8, quantized output")
    finally:
        L.llmq_gemm_force_plan(-1, 1)
    acc = R.int8_gemm_exact(qx[:, :K].contiguous(), qw[:, :K].contiguous())
    assert torch.equal(dump.cpu(), acc)
    want = R.w8a8_epilogue_per_token_per_channel(acc, sx, sw, bias, torch.bfloat16)
    assert torch.equal(y[:, :N].cpu().view(torch.int16), want.view(torch.int16))
    for r in (y, *f8, quant):
        assert (r[:, N:] == 7.0).all()
    for r, x in zip(f8, (a, a5)):
        prod = x[:, :K].double() @ b[:, :K].double().t() * sx.double().view(-1, 1) * sw.double()
        ref = prod + bias.double()
        assert ((r[:, :N].cpu().double() - ref).abs() <= 2e-4 * prod.abs().max() + ref.abs() / 256).all()
    padded = torch.nn.functional.pad(f8[0][:, :N], (0, -N % 8))  # the quantizer takes rows of whole 16 bytes
    assert torch.equal(quant[:, :N], static_per_tensor_quantize(padded, scale.view(1)).to(torch.bfloat16).float()[:, :N] * scale)


# blocks that go from one group of 64 or 32 channels to the next: a block has one or two, three, more than sixteen at one block a CU (then there are more blocks), with
# one stage, several, a ragged end, and channels that end inside the last group
@pytest.mark.parametrize("M,N,K", [(16, 16400, 528), (3, 36904, 3600), (1, 270016, 256), (9, 33000, 2048)])
@pytest.mark.parametrize("variant", [12, 13])
def test_many_groups_of_channels(cuda, variant, M, N, K):
    from llmqrt_amd import _abi
    L = _abi.lib()
    g = torch.Generator().manual_seed(N)
    qx, qw = _ints((M, K), M), _ints((N, K), N)
    sx, sw = torch.rand(M, generator=g) * 0.01 + 1e-3, torch.rand(N, generator=g) * 0.01 + 1e-3
    bias = torch.randn(N, generator=g).bfloat16()
    dev = [t.to(cuda) for t in (sx, sw, bias, qx, qw)]
    p = [t.data_ptr() for t in dev]
    out = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device=cuda)
    _abi.check(L.llmq_gemm_force_plan(110 + variant, 1), "force_plan")
    try:
        _abi.check(L.llmq_gemm_w8a8(p[3], K, p[4], K, p[0], p[1], 1.0, None, p[2], 0, 1.0, out.data_ptr(), 0, N, M, N, K, None, None, 0,
                                    torch.cuda.current_stream().cuda_stream), "int8")
    finally:
        L.llmq_gemm_force_plan(-1, 1)
    acc = (qx.double() @ qw.double().t()).int()  # exact: fewer than 2^53
    want = R.w8a8_epilogue_per_token_per_channel(acc, sx, sw, bias, torch.bfloat16)
    assert torch.equal(out[:M].cpu().view(torch.int16), want.view(torch.int16)) and (out[M] == 7.0).all()


# the same with fp8 operands and the other forms of the epilogue: e4m3 and e5m2 activations, one scale for the tensor read from the device and none per row or
# channel, fp16 results, the quantized fp32 output, raw sums, rows and outputs further apart than they are long
@pytest.mark.parametrize("M,N,K", [(16, 16400, 528), (3, 36904, 1040), (5, 33000, 2048)])
@pytest.mark.parametrize("variant", [12, 13])
def test_many_groups_fp8_and_every_epilogue(cuda, variant, M, N, K):
    from llmqrt_amd import _abi
    from llmqrt_amd.quantize import static_per_tensor_quantize
    L = _abi.lib()
    ld, ldo = K + 32, N + 8
    g = torch.Generator().manual_seed(N + K)
    a, b = [(torch.randn(n, ld, generator=g) * 30).clamp(-448, 448).to(torch.float8_e4m3fn).to(cuda) for n in (M, N)]
    a5 = a.float().to(torch.float8_e5m2)
    qx, qw = _ints((M, ld), M).to(cuda), _ints((N, ld), N).to(cuda)
    sx, sw = (torch.rand(M, generator=g) * 0.01 + 1e-3).to(cuda), (torch.rand(N, generator=g) * 0.01 + 1e-3).to(cuda)
    alpha, bias = torch.tensor([3e-4], device=cuda), torch.randn(N, generator=g).bfloat16().to(cuda)
    stream = torch.cuda.current_stream().cuda_stream
    names = {torch.bfloat16: 0, torch.float16: 1}

    def fp8(x, fmt, rows, channels, scalar, out_dtype, dump=None):
        out = torch.full((M, ldo), 7.0, dtype=out_dtype, device=cuda)
        _abi.check(L.llmq_gemm_fp8(x.data_ptr(), fmt, ld, b.data_ptr(), ld, _abi.ptr(rows), _abi.ptr(channels), 1.0, _abi.ptr(scalar), bias.data_ptr(), 0, 1.0,
                                   out.data_ptr(), names[out_dtype], ldo, M, N, K, _abi.ptr(dump), None, 0, stream), "fp8")
        assert bool((out[:, N:] == 7.0).all())
        return out[:, :N]
    _abi.check(L.llmq_gemm_force_plan(110 + variant, 1), "force_plan")
    try:
        dump, dump8 = torch.full((M, N), -1, dtype=torch.int32, device=cuda), torch.full((M, N), -1.0, device=cuda)
        token = fp8(a, 0, sx, sw, None, torch.bfloat16, dump8)
        wide = fp8(a5, 1, sx, sw, None, torch.bfloat16)
        tensor = fp8(a, 0, None, None, alpha, torch.float16)
        i8 = torch.full((M, ldo), 7.0, dtype=torch.float16, device=cuda)
        _abi.check(L.llmq_gemm_w8a8(qx.data_ptr(), ld, qw.data_ptr(), ld, None, None, 1.0, alpha.data_ptr(), bias.data_ptr(), 0, 1.0, i8.data_ptr(), 1, ldo, M, N, K,
                                    dump.data_ptr(), None, 0, stream), "int8")
        scale = tensor.float().abs().max().view(1) / 300
        quant = torch.full((M, ldo), 7.0, device=cuda)
        _abi.check(L.llmq_gemm_fp8_quantized_output(a.data_ptr(), 0, ld, b.data_ptr(), ld, None, None, 1.0, alpha.data_ptr(), bias.data_ptr(), 0, 1.0, scale.data_ptr(),
                                                    quant.data_ptr(), 1, ldo, M, N, K, None, 0, stream), "quantized output")
    finally:
        L.llmq_gemm_force_plan(-1, 1)
    prod, prod5 = (x[:, :K].double() @ b[:, :K].double().t() for x in (a, a5))
    per = sx.double().view(-1, 1) * sw.double()
    for got, p, scales, half_ulp in ((token, prod, per, 2.0 ** -9), (wide, prod5, per, 2.0 ** -9), (tensor, prod, alpha.double(), 2.0 ** -12)):
        p = p * scales
        ref = p + bias.double()
        # exact products; what the matrix cores' accumulation window loses, fp32 sums, one rounding to the output type
        assert bool(((got.double() - ref).abs() <= 2e-4 * p.abs().max() + 2 * half_ulp * ref.abs()).all())
    assert bool(((dump8.double() - prod).abs() <= 2e-4 * prod.abs().max()).all())
    acc = qx[:, :K].double() @ qw[:, :K].double().t()
    assert torch.equal(dump, acc.int())
    want = (acc.float().double() * alpha.double() + bias.double()).float().half()  # one fma, then the output type
    assert torch.equal(i8[:, :N], want)
    padded = torch.nn.functional.pad(tensor, (0, -N % 8))
    assert torch.equal(quant[:, :N], static_per_tensor_quantize(padded, scale).to(torch.float16).float()[:, :N] * scale) and bool((quant[:, N:] == 7.0).all())


# fp8 on both sides of the planner's lines of channels
@pytest.mark.parametrize("M,N,K", [(7, 8192, 2048), (7, 8200, 2048), (7, 16384, 1024), (7, 16392, 1040), (7, 20480, 8192), (7, 20488, 1536), (7, 24576, 2048), (7, 24584, 2048),
                                   (7, 32776, 1152), (7, 29256, 1152)])
def test_planned_fp8(cuda, M, N, K):
    from llmqrt_amd.sq_fp8_kernels import cutlass_f8f8bf16_rowwise_sm89
    g = torch.Generator().manual_seed(M + N)
    a, b = [(torch.randn(n, K, generator=g) * 30).clamp(-448, 448).to(torch.float8_e4m3fn).to(cuda) for n in (M, N)]
    sx, sw = (torch.rand(M, generator=g) * 0.01 + 1e-3).to(cuda), (torch.rand(N, generator=g) * 0.01 + 1e-3).to(cuda)
    y = cutlass_f8f8bf16_rowwise_sm89(a, b.t(), None, sx.view(-1, 1), sw.view(1, -1), True)
    ref = a.double() @ b.double().t() * sx.double().view(-1, 1) * sw.double()
    assert bool(((y.double() - ref).abs() <= 2e-4 * ref.abs().max() + 2.0 ** -8 * ref.abs()).all())


# what the planner itself picks on both sides of its limits: tokens, K and channels
@pytest.mark.parametrize("M,N,K", [(1, 3584, 3584), (16, 4104, 2048), (16, 4088, 2048), (17, 3584, 3584), (32, 4608, 3584), (33, 4608, 3584), (48, 4608, 3584),
                                   (64, 3584, 3584), (65, 3584, 3584), (8, 896, 4864), (32, 896, 1024), (32, 896, 1152), (20, 16128, 2048), (16, 1024, 18944),
                                   (16, 8192, 1152), (16, 8200, 1152), (16, 8200, 768), (5, 16392, 1024), (4, 24584, 1024)])
def test_planned(cuda, M, N, K):
    from llmqrt_amd.sq_fp8_kernels import w8a8_int8_linear_bbf16_obf16_per_channel
    g = torch.Generator().manual_seed(M + N)
    qx, qw = _ints((M, K), M), _ints((N, K), N + 1)
    sx, sw = torch.rand(M, generator=g) * 0.01 + 1e-3, torch.rand(N, generator=g) * 0.01 + 1e-3
    bias = torch.randn(N, generator=g).bfloat16()
    y = w8a8_int8_linear_bbf16_obf16_per_channel(qx.to(cuda), qw.to(cuda).t(), bias.to(cuda), sx.to(cuda).view(-1, 1), sw.to(cuda).view(1, -1))
    want = R.w8a8_epilogue_per_token_per_channel(R.int8_gemm_exact(qx, qw), sx, sw, bias, torch.bfloat16)
    assert torch.equal(y.cpu().view(torch.int16), want.view(torch.int16))
