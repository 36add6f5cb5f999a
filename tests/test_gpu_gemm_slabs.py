"""Few-token GEMM in slabs of tokens (17 and more tokens, few channels) and the tiles of whole 128-byte lines, at the edges of slabs, tiles and
of the sizes where the planner lets them compete."""
import pytest
import torch

from oracle import ref_math as R

pytestmark = pytest.mark.gpu

# what the planner picks on both sides of its token and channel limits, ragged channels, short and long K (slabs of 16 tokens, 32 for int8 at
# 128 tokens and more, one block row, tiles); every slab variant is forced further down
SHAPES = [(60, 640, 1664), (40, 1152, 6528), (45, 1160, 1280), (17, 520, 2048), (33, 1000, 1536), (65, 768, 1664), (82, 776, 1664),
          (128, 2048, 896), (129, 1024, 896), (200, 512, 3584), (256, 1024, 1024), (257, 1024, 1024), (5, 1024, 18944), (64, 8192, 896)]


def _ints(shape, seed, dtype=torch.int8):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(-127, 128, shape, generator=g, dtype=torch.int32).to(dtype)


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int8_accumulators_exact(cuda, M, N, K):
    from llmqrt_amd.sq_fp8_kernels import w8a8_int8_linear_bbf16_obf16_per_channel
    g = torch.Generator().manual_seed(M + N)
    qx, qw = _ints((M, K), M), _ints((N, K), N)
    sx, sw = torch.rand(M, generator=g) * 0.01 + 1e-3, torch.rand(N, generator=g) * 0.01 + 1e-3
    bias = torch.randn(N, generator=g).bfloat16()
    acc = R.int8_gemm_exact(qx, qw)
    dump = torch.full((M, N), -1, dtype=torch.int32, device=cuda)
    args = (qx.to(cuda), qw.to(cuda).t(), bias.to(cuda), sx.to(cuda).view(-1, 1), sw.to(cuda).view(1, -1))
    y = w8a8_int8_linear_bbf16_obf16_per_channel(*args, _acc_dump=dump)
    assert torch.equal(dump.cpu(), acc)
    ref = R.w8a8_epilogue_per_token_per_channel(acc, sx, sw, bias, torch.bfloat16)
    assert torch.equal(y.cpu().view(torch.int16), ref.view(torch.int16))
    assert torch.equal(w8a8_int8_linear_bbf16_obf16_per_channel(*args).view(torch.int16), y.view(torch.int16))


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_fp8_with_and_without_output_quantization(cuda, M, N, K):
    """The GEMM against float64 (fp8 products are exact; 2e-4 of the largest is what the matrix cores' accumulation window loses, half a
    bf16 step the output), then its quantized output against the three steps on that GEMM result, bit for bit."""
    from llmqrt_amd.quantize import static_per_tensor_quantize
    from llmqrt_amd.sq_fp8_kernels import cutlass_f8f8bf16_tensorwise_sm89, f8f8_tensorwise_quantized_output
    g = torch.Generator().manual_seed(M * N)
    a = (torch.randn(M, K, generator=g) * 30).clamp(-448, 448).to(torch.float8_e4m3fn)
    b = (torch.randn(N, K, generator=g) * 30).clamp(-448, 448).to(torch.float8_e4m3fn)
    bias = (50 * torch.randn(N, generator=g)).bfloat16()
    alpha = torch.tensor(0.01)
    ref = a.double() @ b.double().t() * 0.01 + bias.double()
    y = cutlass_f8f8bf16_tensorwise_sm89(a.to(cuda), b.to(cuda).t(), bias.to(cuda), alpha.to(cuda), 1.0, "bfloat16")
    assert ((y.cpu().double() - ref).abs() <= 2e-4 * ref.abs().max() + ref.abs() / 256).all()
    scale = torch.tensor([float(ref.abs().max()) / 300], device=cuda)
    q = static_per_tensor_quantize(y, scale)
    want = q.to(torch.bfloat16).float() * scale
    got = f8f8_tensorwise_quantized_output(a.to(cuda), b.to(cuda).t(), bias.to(cuda), alpha.to(cuda), 1.0, "bfloat16", scale)
    assert got.dtype == torch.float32 and torch.equal(got, want)


@pytest.mark.parametrize("slab", [16, 32, 64])
@pytest.mark.parametrize("variant", range(6))
@pytest.mark.parametrize("last", ["one row", "ragged", "full"])
def test_every_slab_variant(cuda, slab, variant, last):
    """1 + (variant & 1) channel tiles per wavefront, 4 << (variant >> 1) wavefronts along a K that ends inside a step, ragged channels: int8
    bit for bit against the exact accumulators, fp8 against float64, its quantized output bit for bit against the steps on the GEMM result."""
    from llmqrt_amd import _abi
    from llmqrt_amd.quantize import static_per_tensor_quantize
    from llmqrt_amd.sq_fp8_kernels import cutlass_f8f8bf16_tensorwise_sm89, f8f8_tensorwise_quantized_output, w8a8_int8_linear_bbf16_obf16_per_channel
    M, N, K = {"one row": slab + 1, "ragged": 2 * slab + slab // 2 - 3, "full": 2 * slab}[last], 328, 1168
    g = torch.Generator().manual_seed(M)
    qx, qw = _ints((M, K), M), _ints((N, K), N)
    sx, sw = torch.rand(M, generator=g) * 0.01 + 1e-3, torch.rand(N, generator=g) * 0.01 + 1e-3
    bias = torch.randn(N, generator=g).bfloat16()
    acc = R.int8_gemm_exact(qx, qw)
    a, b = [(torch.randn(n, K, generator=g) * 30).clamp(-448, 448).to(torch.float8_e4m3fn) for n in (M, N)]
    ref = a.double() @ b.double().t() * 0.01 + bias.double()
    scale = torch.tensor([float(ref.abs().max()) / 300], device=cuda)
    alpha = torch.tensor(0.01, device=cuda)
    dump = torch.full((M, N), -1, dtype=torch.int32, device=cuda)
    L = _abi.lib()
    _abi.check(L.llmq_gemm_force_plan(100 + variant, slab), "force_plan")
    try:
        y = w8a8_int8_linear_bbf16_obf16_per_channel(qx.to(cuda), qw.to(cuda).t(), bias.to(cuda), sx.to(cuda).view(-1, 1),
                                                     sw.to(cuda).view(1, -1), _acc_dump=dump)
        y8 = cutlass_f8f8bf16_tensorwise_sm89(a.to(cuda), b.to(cuda).t(), bias.to(cuda), alpha, 1.0, "bfloat16")
        got = f8f8_tensorwise_quantized_output(a.to(cuda), b.to(cuda).t(), bias.to(cuda), alpha, 1.0, "bfloat16", scale)
    finally:
        L.llmq_gemm_force_plan(-1, 1)
    assert torch.equal(dump.cpu(), acc)
    want = R.w8a8_epilogue_per_token_per_channel(acc, sx, sw, bias, torch.bfloat16)
    assert torch.equal(y.cpu().view(torch.int16), want.view(torch.int16))
    assert ((y8.cpu().double() - ref).abs() <= 2e-4 * ref.abs().max() + ref.abs() / 256).all()
    assert torch.equal(got, static_per_tensor_quantize(y8, scale).to(torch.bfloat16).float() * scale)


@pytest.mark.parametrize("cfg", [4, 5, 8, 9, 10])
@pytest.mark.parametrize("M,N,K", [(192, 128, 128), (193, 256, 256), (384, 384, 384), (127, 136, 512), (576, 120, 1152)])
@pytest.mark.parametrize("splits", [1, 2])
def test_tiles_of_whole_lines(cuda, cfg, M, N, K, splits):
    """One to nine K tiles (fewer and more than LDS stages), interior and edge tiles of the block-wide epilogue, fp16 output with bias."""
    from llmqrt_amd import _abi
    from llmqrt_amd.sq_fp8_kernels import w8a8_int8_linear_bbf16_obf16_per_channel
    if K // splits < 128:
        pytest.skip("a split holds at least one K tile")
    qx, qw = _ints((M, K), 1), _ints((N, K), 2)
    g = torch.Generator().manual_seed(3)
    sx, sw, bias = torch.rand(M, generator=g) * 1e-3, torch.rand(N, generator=g) * 1e-2, torch.randn(N, generator=g).half()
    ref = R.w8a8_epilogue_per_token_per_channel(R.int8_gemm_exact(qx, qw), sx, sw, bias, torch.float16)
    L = _abi.lib()
    _abi.check(L.llmq_gemm_force_plan(cfg, splits), "force_plan")
    try:
        y = w8a8_int8_linear_bbf16_obf16_per_channel(qx.to(cuda), qw.to(cuda).t(), bias.to(cuda), sx.to(cuda).view(-1, 1),
                                                     sw.to(cuda).view(1, -1))
    finally:
        L.llmq_gemm_force_plan(-1, 1)
    assert torch.equal(y.cpu().view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("cfg", [4, 5, 6, 7, 8, 9, 10])
@pytest.mark.parametrize("M,N,K", [(65, 136, 16), (192, 128, 112), (300, 264, 144), (256, 256, 272), (130, 512, 1264), (257, 384, 2032)])
def test_ragged_tail_behind_direct_loads(cuda, cfg, M, N, K):
    """K that ends inside a 128-byte tile: no whole tile, one, a few and more than LDS stages in front of tails of 16 to 112 bytes, without
    a split and with the tail in the last of two, against the register-staged loop bit for bit and the exact accumulators."""
    from llmqrt_amd import _abi
    from llmqrt_amd.sq_fp8_kernels import cutlass_f8f8bf16_rowwise_sm89, w8a8_int8_linear_bbf16_obf16_per_channel
    qx, qw = _ints((M, K), 1), _ints((N, K), 2)
    g = torch.Generator().manual_seed(3)
    sx, sw = torch.rand(M, generator=g) * 1e-3, torch.rand(N, generator=g) * 1e-2
    ref = R.w8a8_epilogue_per_token_per_channel(R.int8_gemm_exact(qx, qw), sx, sw, None, torch.bfloat16)
    a8 = (torch.randn(M, K, generator=g) * 20).to(torch.float8_e4m3fn).to(cuda)
    b8 = (torch.randn(N, K, generator=g) * 20).to(torch.float8_e4m3fn).to(cuda)
    zero = torch.zeros(N, dtype=torch.bfloat16, device=cuda)
    L = _abi.lib()
    try:
        for splits in (1, 2):
            if K // splits < 128 and splits > 1:
                continue
            f8 = []
            for force in (cfg, cfg | 64):
                _abi.check(L.llmq_gemm_force_plan(force, splits), "force_plan")
                y = w8a8_int8_linear_bbf16_obf16_per_channel(qx.to(cuda), qw.to(cuda).t(), zero, sx.to(cuda).view(-1, 1), sw.to(cuda).view(1, -1))
                assert torch.equal(y.cpu().view(torch.int16), ref.view(torch.int16))
                f8.append(cutlass_f8f8bf16_rowwise_sm89(a8, b8.t(), None, sx.to(cuda).view(-1, 1), sw.to(cuda).view(1, -1), True))
            assert torch.equal(f8[0].view(torch.int16), f8[1].view(torch.int16))
    finally:
        L.llmq_gemm_force_plan(-1, 1)


# sizes that the rules of 16 .. 128 rows serve without partial sums, or with fewer than the plan that a full workspace gets
@pytest.mark.parametrize("kind,M,N,K,kept", [("int8", 5, 136, 13056, 0), ("int8", 66, 3896, 5120, 2057088), ("fp8", 98, 2280, 3584, 0),
                                             ("fp8", 5, 2392, 15488, 621920), ("f16", 66, 128, 1152, 0), ("f16", 102, 1320, 10752, 2692800)])
def test_workspace_of_the_rules_is_still_enough(cuda, kind, M, N, K, kept):
    """A caller that kept the workspace size of the rules' plan, or has none where that needs none: the call runs and gives what the GEMM
    with a full workspace gives (int8 bit for bit; fp32 sums in another order: half a bf16 step of the value plus what test_fp8_.. allows)."""
    from llmqrt_amd import _abi
    L = _abi.lib()
    g = torch.Generator().manual_seed(N)
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "int8":
        a, b = _ints((M, K), 1), _ints((N, K), 2)
        ref = R.int8_gemm_exact(a, b).float() * 2.0 ** -10
        query = L.llmq_gemm_workspace_bytes(M, N, K)
    elif kind == "fp8":
        a, b = [(torch.randn(n, K, generator=g) * 30).clamp(-448, 448).to(torch.float8_e4m3fn) for n in (M, N)]
        ref = a.double() @ b.double().t() * 2.0 ** -10
        query = L.llmq_gemm_fp8_quantized_output_workspace_bytes(M, N, K)  # the fp8 plan's own
    else:
        a, b = torch.randn(M, K, generator=g).half(), torch.randn(N, K, generator=g).half()
        ref = a.double() @ b.double().t() * 2.0 ** -10
        query = L.llmq_gemm_f16_workspace_bytes(M, N, K)
    a, b = a.to(cuda), b.to(cuda)

    def run(nbytes):
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=cuda)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=cuda) if nbytes else None
        tail = (out.data_ptr(), _abi.BF16, N, M, N, K, None, _abi.ptr(ws), nbytes, stream)
        if kind == "int8":
            rc = L.llmq_gemm_w8a8(a.data_ptr(), K, b.data_ptr(), K, None, None, 2.0 ** -10, None, None, 0, 0.0, *tail)
        elif kind == "fp8":
            rc = L.llmq_gemm_fp8(a.data_ptr(), _abi.E4M3, K, b.data_ptr(), K, None, None, 2.0 ** -10, None, None, 0, 0.0, *tail)
        else:
            rc = L.llmq_gemm_f16(a.data_ptr(), K, b.data_ptr(), K, 2.0 ** -10, None, 0, 0.0, *tail)
        _abi.check(rc, kind)
        return out.cpu()
    full, small = run(query), run(kept)
    if kind == "int8":
        assert torch.equal(small.view(torch.int16), full.view(torch.int16))
        assert torch.equal(small.view(torch.int16), ref.to(torch.bfloat16).view(torch.int16))
    else:
        for y in (full, small):
            assert ((y.double() - ref).abs() <= 2e-4 * ref.abs().max() + ref.abs() / 256).all()
