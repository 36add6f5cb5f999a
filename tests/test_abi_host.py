"""CPU-only checks of the boundary: the shared library loads, exports every symbol that
include/llmq.h declares, its argument validation returns the documented codes before any HIP
call, and the Python wrappers mirror the reference's interface and error behaviour."""
import ctypes
import pathlib
import re

import pytest
import torch

ROOT = pathlib.Path(__file__).resolve().parent.parent


def _declared_symbols():
    text = (ROOT / "include" / "llmq.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(llmq_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from llmqrt_amd import _abi
    lib = _abi.lib()
    declared = _declared_symbols()
    assert len(declared) >= 14
    for name in declared:
        assert hasattr(lib, name), f"{name} is declared in llmq.h but not exported"
    assert sorted(_abi.SIGNATURES) == declared, "ctypes table and header disagree"
    assert lib.llmq_abi_version() == 1
    assert lib.llmq_status_string(0) == b"ok"
    assert b"workspace" in lib.llmq_status_string(-4)


def test_argument_validation_needs_no_gpu():
    from llmqrt_amd import _abi
    L = _abi.lib()
    buf = ctypes.create_string_buffer(4096)
    p = ctypes.addressof(buf)
    p16 = (p + 15) & ~15
    # negative sizes / misaligned K / strides
    assert L.llmq_gemm_w8a8(p16, 64, p16, 64, None, None, 1.0, None, None, 0, 0.0, p16, 0, 8, -1, 8, 64, None, None, 0, None) == -3
    assert L.llmq_gemm_w8a8(p16, 24, p16, 24, None, None, 1.0, None, None, 0, 0.0, p16, 0, 8, 4, 8, 24, None, None, 0, None) == -3
    assert L.llmq_gemm_w8a8(None, 64, p16, 64, None, None, 1.0, None, None, 0, 0.0, p16, 0, 8, 4, 8, 64, None, None, 0, None) == -1
    assert L.llmq_gemm_w8a8(p16, 64, p16, 64, None, None, 1.0, None, None, 0, 0.0, p16, 2, 8, 4, 8, 64, None, None, 0, None) == -2
    assert L.llmq_gemm_w8a8(p16 + 1, 64, p16, 64, None, None, 1.0, None, None, 0, 0.0, p16, 0, 8, 4, 8, 64, None, None, 0, None) == -6
    assert L.llmq_gemm_w8a8(p16, 64, p16, 64, None, None, 1.0, None, None, 0, 0.0, p16, 0, 8, 0, 8, 64, None, None, 0, None) == 0  # M == 0
    assert L.llmq_gemm_fp8(p16, 7, 64, p16, 64, None, None, 1.0, None, None, 0, 0.0, p16, 0, 8, 4, 8, 64, None, None, 0, None) == -2
    assert L.llmq_quant_i8_per_token(p16, 2, 4, 64, 64, p16, p16, 2, None) == -2      # fp32 activations unsupported
    assert L.llmq_quant_i8_per_token(p16, 0, 4, 60, 64, p16, p16, 0, None) == -3      # K % 8
    assert L.llmq_quant_i8_per_token(p16, 0, 0, 64, 64, p16, p16, 0, None) == 0       # M == 0
    assert L.llmq_quant_i8_per_tensor(p16, 0, 4, 64, 64, p16, p16, 0, None, 0, None) == -4
    assert L.llmq_awq_gemm(p16, 100, p16, p16, p16, None, p16, 2, 64, 100, 128, None, 0, None) == -3   # K % 32
    assert L.llmq_awq_gemm(p16, 128, p16, p16, p16, None, p16, 2, 60, 128, 128, None, 0, None) == -3   # N % 8
    assert L.llmq_awq_dequant(p16, p16, p16, p16, 128, 64, 48, None) == -3                              # K % G
    assert L.llmq_gemm_force_plan(99, 1) == -3 and L.llmq_gemm_force_plan(106, 1) == -3 and L.llmq_gemm_force_plan(-1, 1) == 0
    assert L.llmq_quant_workspace_bytes() >= 4096
    # split-K plans ask for a workspace, plain ones do not
    assert L.llmq_gemm_workspace_bytes(8192, 37888, 3584) == 0
    assert L.llmq_awq_gemm_workspace_bytes(1, 4608, 3584) > 0


# (fp8, M, N, K, whether the row-streaming kernel runs): both sides of the lines beyond which the kernels before it were measured ahead: many tokens of few
# channels over a long and a short K, more channels than 17-64 tokens stream, short rows that leave the last stage empty, rows that fall on few
# memory channels
@pytest.mark.parametrize("fp8,M,N,K,rows", [
    (0, 61, 960, 8704, False), (0, 61, 2560, 4096, True), (0, 50, 512, 9104, False), (0, 50, 512, 7216, True), (1, 57, 952, 1920, False), (1, 57, 2304, 1920, True),
    (0, 49, 9400, 1984, False), (0, 30, 9400, 1984, True), (1, 57, 968, 4096, False), (0, 20, 16808, 1280, False), (0, 20, 16128, 1280, True),
    (0, 22, 1080, 15296, False), (1, 1, 29256, 1152, False), (1, 1, 29256, 1024, True), (1, 1, 29256, 1280, True), (0, 2, 14408, 11008, False), (0, 2, 14408, 10752, True),
    (0, 7, 25576, 8192, False), (1, 7, 25576, 8192, True), (0, 4, 22384, 16384, False), (0, 2, 30896, 4096, False), (0, 16, 34104, 8192, True),
    (1, 8, 8512, 20480, False), (1, 2, 20544, 16384, False), (1, 2, 14408, 16384, True), (1, 1, 2760, 3456, False), (1, 8, 2760, 3456, True), (0, 1, 3624, 11008, False),
    (0, 2, 7984, 16384, False), (0, 2, 7984, 14336, True), (0, 1, 37888, 3584, True), (0, 16, 3584, 3584, True), (0, 65, 3584, 3584, False)])
def test_few_token_gemm_lines(fp8, M, N, K, rows):
    from llmqrt_amd import _abi
    cfg = _abi.lib().llmq_gemm_planned_config(fp8, M, N, K)
    assert (110 <= cfg <= 123) == rows, cfg


# bytes that the kernel which runs uses (0: one launch or one split), whether it needs arrival counters; llmq_awq_gemm_partials_bytes covers every kernel a
# size may run and is larger for some of these: an fp16 call of a small group that does not stream, a prompt that streams in one launch.  Few weights past 64
# tokens are split, which a plan over eight stages and more in one launch loses to
@pytest.mark.parametrize("bf16,M,N,K,group,some,counters", [
    (0, 1, 3584, 3584, 128, True, 1), (1, 1, 3584, 3584, 128, True, 1), (0, 64, 3584, 18944, 128, True, 0), (0, 12, 1152, 896, 32, False, 0),
    (1, 12, 1152, 896, 32, True, 0), (0, 148, 632, 512, 32, True, 0), (0, 79, 1560, 512, 32, True, 0), (0, 777, 2048, 1024, 128, False, 0), (1, 96, 4608, 896, 32, False, 0), (0, 200, 1152, 3552, 32, True, 0)])
def test_awq_linear_workspace(bf16, M, N, K, group, some, counters):
    from llmqrt_amd import _abi
    L, flag = _abi.lib(), ctypes.c_int(7)
    need = L.llmq_awq_linear_partials_bytes(_abi.BF16 if bf16 else _abi.F16, M, N, K, group, K, ctypes.byref(flag))
    assert (need > 0) == some and flag.value == counters
    assert need <= L.llmq_awq_gemm_partials_bytes(M, N, K, group)


# (bf16, tokens, channels, K, group, kernel: s streaming tiles, f few-token, r register-streaming, t tiles): both sides of the lines between the kernels; group 128
# with channels off the few-token kernel's grid of 32 among them
@pytest.mark.parametrize("bf16,M,N,K,group,kernel", [
    (0, 35, 3792, 768, 128, "r"), (0, 62, 3624, 1024, 128, "r"), (0, 29, 13576, 1024, 128, "s"), (1, 35, 3792, 768, 128, "s"), (0, 35, 3792, 768, 64, "s"),
    (0, 1, 32776, 7424, 128, "r"), (0, 10, 31800, 7296, 128, "r"), (0, 10, 33800, 7296, 128, "s"), (0, 7, 33296, 7040, 128, "r"), (0, 5, 14088, 17408, 128, "s"), (0, 5, 11768, 17408, 128, "s"), (0, 1, 9904, 17792, 128, "r"),
    (0, 8, 11768, 17408, 128, "s"), (0, 42, 616, 10624, 128, "s"), (0, 39, 9744, 896, 128, "r"), (1, 2, 36208, 7552, 128, None), (1, 3, 36208, 7552, 128, "s"), (0, 1, 32768, 7424, 128, "f"), (0, 18, 4992, 1024, 128, "f"), (0, 37, 896, 896, 128, "s"), (0, 60, 256, 3584, 128, "f"),
    (0, 64, 37888, 3584, 128, "s"), (0, 65, 896, 896, 32, "s"), (0, 65, 896, 992, 32, "t"), (0, 8, 4096, 4096, 64, "r"), (0, 8, 8192, 4096, 64, "s")])
def test_awq_lines(bf16, M, N, K, group, kernel):
    from llmqrt_amd import _abi
    L, dt = _abi.lib(), _abi.BF16 if bf16 else _abi.F16
    cfg = L.llmq_awq_planned_config(dt, M, N, K, group, K)
    if kernel is None:  # the module converts around the fp16 kernel
        assert cfg == -2 and not L.llmq_awq_linear_bf16_supported(M, N, K, group, K)
        return
    assert kernel == ("s" if cfg >= 12 else "f" if cfg == 8 else "t" if cfg in (3, 4, 7) else "r" if cfg == 1 else "?"), cfg


# kind (0 int8 per token, 1 fp8 per token, 2 int8 per tensor, 3 fp8 per tensor, 4 static), tokens, channels, K, one launch from a program's loop, in a graph
@pytest.mark.parametrize("kind,M,N,K,loop,graph", [
    (2, 16, 896, 4864, 1, 0), (3, 14, 416, 4096, 1, 0), (3, 10, 896, 3072, 1, 1), (2, 9, 232, 6160, 0, 0), (2, 2, 312, 17408, 0, 0), (2, 1, 3584, 18944, 1, 1),
    (3, 8, 896, 8192, 0, 0), (3, 9, 896, 8192, 0, 0), (2, 1, 3584, 3584, 1, 1), (2, 1, 37888, 3584, 1, 0), (3, 2, 8704, 6464, 0, 0), (3, 1, 14200, 13088, 0, 0),
    (3, 16, 9728, 896, 1, 1), (0, 5, 688, 7936, 0, 0), (0, 5, 688, 1600, 1, 1), (1, 10, 3584, 3584, 1, 0), (1, 2, 3584, 3584, 1, 1), (0, 4, 3584, 7936, 1, 0),
    (0, 2, 22368, 400, 1, 1), (0, 3, 18064, 1600, 1, 1), (0, 2, 22368, 384, 0, 0), (1, 4, 37504, 1408, 0, 0), (4, 8, 3584, 3584, 1, 0), (4, 4, 3584, 3584, 1, 1),
    (4, 17, 64, 64, 0, 0), (5, 1, 64, 64, 0, 0)])
def test_one_launch_lines(kind, M, N, K, loop, graph):
    from llmqrt_amd import _abi
    L = _abi.lib()
    assert (L.llmq_linear_one_launch_preferred(kind, M, N, K), L.llmq_linear_one_launch_ahead(kind, M, N, K)) == (loop, graph)


@pytest.mark.parametrize("kind", range(5))
def test_one_launch_lines_have_no_holes(kind):
    """More tokens of the same sizes make more codes for every block: a size that takes two launches takes two with more tokens as well."""
    from llmqrt_amd import _abi
    L = _abi.lib()
    for line in (L.llmq_linear_one_launch_preferred, L.llmq_linear_one_launch_ahead):
        for N in (64, 896, 1024, 1032, 3584, 4096, 4104, 8192, 9728, 16384, 37888):
            for K in (64, 896, 1888, 1904, 3584, 4864, 5120, 5136, 6144, 8192, 18944):
                taken = [line(kind, M, N, K) for M in range(1, 18)]
                assert taken == sorted(taken, reverse=True), (N, K, taken)


def test_planned_config_refuses():
    from llmqrt_amd import _abi
    awq = _abi.lib().llmq_awq_planned_config
    assert awq(_abi.F16, 4, 64, 100, 100, 100) == awq(_abi.F16, 4, 60, 128, 128, 128) == awq(_abi.F16, 0, 64, 128, 128, 128) == -3
    plan = _abi.lib().llmq_gemm_planned_config
    assert plan(0, 0, 64, 64) == plan(0, 4, 64, 40) == plan(1, 4, -1, 64) == -3


def test_wrappers_fail_loudly_off_gpu():
    from llmqrt_amd import sq_fp8_kernels as ops
    from llmqrt_amd.quantize import quantize_activation_per_token_absmax
    x = torch.zeros(4, 64, dtype=torch.int8)
    w = torch.zeros(8, 64, dtype=torch.int8)
    with pytest.raises(RuntimeError, match="GPU"):
        ops.w8a8_int8_linear_bbf16_obf16_per_tensor(x, w.t(), torch.zeros(8, dtype=torch.bfloat16), 1.0, 1.0)
    with pytest.raises(RuntimeError, match="GPU"):
        quantize_activation_per_token_absmax(torch.zeros(2, 8, dtype=torch.bfloat16))


def test_missing_library_is_an_error(monkeypatch, tmp_path):
    from llmqrt_amd import _abi
    monkeypatch.setattr(_abi, "_lib", None)
    monkeypatch.setattr(_abi, "_LIB_PATH", tmp_path / "libllmq_gfx950.so")
    with pytest.raises(RuntimeError, match="no CPU or PyTorch fallback"):
        _abi.lib()


def test_product_package_never_touches_the_oracle():
    for path in (ROOT / "llmqrt_amd").rglob("*.py"):
        text = path.read_text()
        assert "oracle" not in text, f"{path} mentions the oracle"


def test_registry_and_module_interfaces():
    from llmqrt_amd.linear import (FP8DynamicLinear, FP8StaticLinear, SqW8A8BBF16OBF16PerTensor, WQLinear_GEMM,
                                   get_concrete_linear_module, method_to_linear)
    assert set(method_to_linear) == {"awq", "sq", "fp8_static_quant", "fp8_dynamic_quant"}
    assert get_concrete_linear_module("awq") is WQLinear_GEMM
    lin = torch.nn.Linear(128, 64, bias=True)
    sq = SqW8A8BBF16OBF16PerTensor.from_linear(lin, 8, 0, True, dtype=torch.bfloat16)
    assert sq.qweight.shape == (64, 128) and sq.qweight.dtype == torch.int8
    assert sq.bias.dtype == torch.bfloat16 and sq.weight_scale.dim() == 0 and sq.input_scale.dim() == 0
    assert set(sq.state_dict()) == {"qweight", "bias", "weight_scale", "input_scale"}
    f8 = FP8DynamicLinear.from_linear(lin, 8, 0, True, dtype=torch.bfloat16, per_tensor=False)
    assert f8.weight.dtype == torch.bfloat16 and f8.weight_scale.shape == (64, 1)
    assert FP8DynamicLinear.from_linear(lin, 8, 0, True, per_tensor=True).weight_scale.shape == (1,)
    st = FP8StaticLinear.from_linear(lin, 8, 0, True)
    assert set(st.state_dict()) == {"weight", "weight_scale", "bias", "input_scale", "output_scale"}
    awq = WQLinear_GEMM.from_linear(lin, 4, 64, True)
    assert awq.qweight.shape == (128, 8) and awq.qzeros.shape == (2, 8) and awq.scales.shape == (2, 64)
    assert awq.scales.dtype == torch.float16 and awq.bias.dtype == torch.float16
    with pytest.raises(AssertionError):
        FP8DynamicLinear.from_linear(lin, 8, 128, True)
    with pytest.raises(NotImplementedError):
        WQLinear_GEMM(8, 64, 128, 64, False, "cpu")


def test_awq_module_packer_matches_oracle():
    """from_linear takes scales / zeros as [K/G, N], the orientation the reference indexes
    (linear_awq.py:165-186, 203-219); N != K/G here so a transposed argument cannot pass unnoticed."""
    from llmqrt_amd.linear import WQLinear_GEMM
    from oracle import ref_math as R
    g = torch.Generator().manual_seed(0)
    lin = torch.nn.Linear(128, 64, bias=False)
    lin.weight.data = 0.02 * torch.randn(64, 128, generator=g)
    G = 64
    wg = lin.weight.data.t().contiguous().view(2, G, 64)      # [K/G, G, N]
    mx, mn = wg.amax(1), wg.amin(1)
    scales = ((mx - mn) / 15).clamp(min=1e-5)                 # [K/G, N]
    zeros = (-mn / scales).round().clamp(0, 15)               # [K/G, N]
    m = WQLinear_GEMM.from_linear(lin, 4, G, False, scales=scales, zeros=zeros)
    assert m.scales.shape == (2, 64) and torch.equal(m.scales, scales.half())
    iw = R.awq_unpack(m.qweight)
    assert iw.min() >= 0 and iw.max() <= 15
    assert torch.equal(R.awq_unpack(m.qzeros), zeros.int())
    # element by element against the reference's loop: intw[k, n] = round((W[n, k] + z s) / s)
    for k, n in [(0, 0), (5, 63), (64, 1), (127, 40)]:
        want = torch.round((lin.weight.data[n, k] + zeros[k // G, n] * scales[k // G, n]) / scales.half()[k // G, n])
        assert iw[k, n] == int(want)
    deq = R.awq_dequantize(m.qweight, m.qzeros, m.scales, G)
    assert (deq.float() - lin.weight.data.t()).abs().max() <= 0.51 * scales.max()
    with pytest.raises(RuntimeError, match="scales and zeros must be"):
        WQLinear_GEMM.from_linear(lin, 4, G, False, scales=scales.t().contiguous(), zeros=zeros.t().contiguous())


def test_workload_shapes_and_byte_counts():
    from llmqrt_amd import workloads as W
    assert W.QWEN2_7B_PROJ["gate_up"] == (3584, 37888) and W.CONFIG0_SHAPE == (16, 896, 4864)
    x = W.activations(16, 896, 0)
    assert x.dtype == torch.bfloat16 and x.shape == (16, 896)
    assert torch.equal(x, W.activations(16, 896, 0))                     # seeded
    assert 15 < x.float().abs().amax(-1).min() < 100                     # outlier channels set the row max
    q, s = W.int8_weights(64, 128, 1)
    assert q.dtype == torch.int8 and s.shape == (64,) and q.abs().amax(1).eq(127).all()
    f, fs = W.fp8_weights(64, 128, 1)
    assert f.dtype == torch.float8_e4m3fn and f.float().abs().amax(1).eq(448).all()
    assert W.gemm_ops(2048, 4608, 3584) == 67645734912
    assert W.awq_gemm_bytes(1, 4608, 3584) == 8596480                    # 8.60 MB
    assert W.w8a8_gemm_bytes(16, 4864, 896) == 4547648                   # 4.55 MB


def test_rmsnorm_argument_validation_needs_no_gpu():
    from llmqrt_amd import _abi
    L = _abi.lib()
    ok_ptr = 0x1000
    # null weight / output, bad dtype, K not a multiple of 8, misaligned input
    assert L.llmq_rmsnorm(ok_ptr, 0, 4, 64, 64, None, 1e-6, ok_ptr, None, None) == -1
    assert L.llmq_rmsnorm(ok_ptr, 0, 4, 64, 64, ok_ptr, 1e-6, None, None, None) == -1
    assert L.llmq_rmsnorm(ok_ptr, 2, 4, 64, 64, ok_ptr, 1e-6, ok_ptr, None, None) == -2
    assert L.llmq_rmsnorm(ok_ptr, 0, 4, 60, 64, ok_ptr, 1e-6, ok_ptr, None, None) == -3
    assert L.llmq_rmsnorm(ok_ptr + 2, 0, 4, 64, 64, ok_ptr, 1e-6, ok_ptr, None, None) == -6
    assert L.llmq_rmsnorm(ok_ptr, 0, 0, 64, 64, ok_ptr, 1e-6, ok_ptr, None, None) == 0
    assert L.llmq_rmsnorm_quant_i8_per_token(ok_ptr, 0, 4, 64, 64, ok_ptr, 1e-6, None, None, ok_ptr, 0, None, None) == -1
    assert L.llmq_rmsnorm_quant_i8_per_token(ok_ptr, 0, 4, 64, 64, ok_ptr, 1e-6, None, ok_ptr, ok_ptr, 1, None, None) == -2
    assert L.llmq_rmsnorm_quant_fp8_per_token(ok_ptr, 1, 4, 64, 32, ok_ptr, 1e-6, None, ok_ptr, ok_ptr, None, None) == -3


def test_bench_refuses_more_than_one_gpu():
    """bench.py measures one GPU; asking for more exits with a message instead of running."""
    import subprocess
    import sys
    root = pathlib.Path(__file__).resolve().parent.parent
    r = subprocess.run([sys.executable, str(root / "bench.py"), "--gpus", "2"], capture_output=True, text=True, timeout=300)
    assert r.returncode != 0
    assert "one GPU" in r.stderr and r.stdout.strip() == ""


@pytest.mark.parametrize("M,N,K", [(2313, 1824, 18288), (410, 21624, 18512), (509, 8528, 16832), (6162, 1440, 18320), (1230, 8088, 19872)])
def test_plans_fit_the_static_scratch(M, N, K):
    """Problems near the line between one pass and a K split, which llmq_gemm_w8a8_static takes in one pass."""
    from llmqrt_amd import _abi
    L = _abi.lib()
    assert L.llmq_gemm_workspace_bytes(M, N, K) <= L.llmq_gemm_static_scratch_bytes()


def test_workspace_figures_by_format():
    """A format's figure is what its own plan splits; the common one covers both.  200 x 512 x 3584 runs in one launch in either format."""
    from llmqrt_amd import _abi
    L = _abi.lib()
    for M, N, K in [(200, 512, 3584), (109, 29600, 6144), (512, 3584, 18944), (1000, 4608, 3600), (71, 3880, 12800), (16, 896, 4864), (0, 8, 16)]:
        i8, f8 = L.llmq_gemm_w8a8_workspace_bytes(M, N, K), L.llmq_gemm_fp8_workspace_bytes(M, N, K)
        assert L.llmq_gemm_workspace_bytes(M, N, K) >= max(i8, f8)
        assert f8 == L.llmq_gemm_fp8_quantized_output_workspace_bytes(M, N, K)
        assert all(b == 0 or (b % (4 * M * N) == 0 and b > 4 * M * N) for b in (i8, f8)), "two or more partial tensors, or none"
    assert L.llmq_gemm_w8a8_workspace_bytes(200, 512, 3584) == 0 == L.llmq_gemm_fp8_workspace_bytes(200, 512, 3584)


def test_repeated_workspace_query_searches_no_plan():
    """A size that is already planned costs what an unsplit one costs (a search takes several times the call itself)."""
    import time
    from llmqrt_amd import _abi
    L = _abi.lib()

    def cost(M, N, K):
        best = float("inf")
        for _ in range(30):
            t = time.perf_counter()
            for _ in range(300):
                L.llmq_gemm_workspace_bytes(M, N, K)
            best = min(best, time.perf_counter() - t)
        return best
    assert cost(512, 3584, 18944) < 2 * cost(8192, 37888, 3584)


def test_first_plan_of_a_size_is_one_search():
    """Every prompt length is a new size for a model's projections.  Where slabs, the table and the rules compete a size is planned in about
    the time of the rounds model's own search (1.2 times through ctypes; with two searches of the table, and the rounds model's beside them, 2.4
    times)."""
    import time
    from llmqrt_amd import _abi
    L = _abi.lib()

    def cost(M, K, first):
        best = float("inf")
        for rep in range(20):
            t = time.perf_counter()
            for i in range(40):
                L.llmq_gemm_fp8_quantized_output_workspace_bytes(M, first + 8 * (40 * rep + i), K)
            best = min(best, time.perf_counter() - t)
        return best
    slabs = min(cost(129 + i, 3584, 256 + 8 * i) for i in range(3))
    rounds = min(cost(129 + i, 20736, 256 + 8 * i) for i in range(3))
    assert slabs < 1.8 * rounds


def _moved_tensors(mod, how):
    """The module's tensors where nn.Module's dictionaries do not hold them under their names."""
    if how == "replica":  # as torch.nn.parallel.replicate leaves a module: parameters are plain attributes
        rep = mod._replicate_for_data_parallel()
        for name, p in mod._parameters.items():
            if p is not None:
                setattr(rep, name, p.detach())
        return rep
    if how == "attributes":
        for store in (mod._parameters, mod._buffers):
            for name in [n for n, t in store.items() if t is not None]:
                t = store.pop(name)
                object.__setattr__(mod, name, t.detach())
        return mod
    for store in (mod._parameters, mod._buffers):
        for name in [n for n, t in store.items() if t is not None and t.is_floating_point()]:
            if store is mod._buffers:
                mod.register_parameter(name, torch.nn.Parameter(store.pop(name), requires_grad=False))
            torch.nn.utils.parametrize.register_parametrization(mod, name, torch.nn.Identity())
    return mod


def _all_modules():
    from llmqrt_amd.linear import (FP8DynamicLinear, FP8StaticLinear, SqW8A8BBF16OBF16PerChannel,
                                   SqW8A8BBF16OBF16PerTensor, WQLinear_GEMM)
    lin = torch.nn.Linear(128, 64, bias=True)
    return {"sq": SqW8A8BBF16OBF16PerTensor.from_linear(lin, 8, 0, True), "sq_channel": SqW8A8BBF16OBF16PerChannel.from_linear(lin, 8, 0, True),
            "fp8": FP8DynamicLinear.from_linear(lin), "fp8_token": FP8DynamicLinear.from_linear(lin, per_tensor=False),
            "static": FP8StaticLinear.from_linear(lin), "static_out": FP8StaticLinear.from_linear(lin, quantize_output=True),
            "awq": WQLinear_GEMM.from_linear(lin, 4, 64, True)}


@pytest.mark.parametrize("how", ["replica", "attributes", "parametrized"])
def test_forward_takes_tensors_that_are_not_registered(how):
    """The general path, which reads the attributes, takes such a module; off the GPU it says so instead of a KeyError."""
    x = torch.zeros(2, 128, dtype=torch.bfloat16)
    for name, mod in _all_modules().items():
        mod = _moved_tensors(mod, how)
        with pytest.raises((RuntimeError, AssertionError)):
            mod(x)
        if name == "sq_channel":
            with pytest.raises(RuntimeError, match="GPU"):
                mod.forward_quantized(x.to(torch.int8), torch.ones(2, 1), torch.bfloat16)
        if name == "fp8_token":
            with pytest.raises(RuntimeError, match="GPU"):
                mod.forward_quantized(x.to(torch.float8_e4m3fn), torch.ones(2, 1))


def test_fp8_copies_follow_a_parametrized_tensor():
    """A parametrization makes a new tensor on each access, often at the address of the one before: the fp8 copy of the
    weight and the flat scales must come from the tensor of this access."""
    class Double(torch.nn.Module):
        def forward(self, t):
            return t * 2

    mod = _all_modules()["fp8_token"]
    for name in ("weight", "weight_scale"):
        torch.nn.utils.parametrize.register_parametrization(mod, name, Double())
    values = [(torch.full((64, 128), float(i)), torch.full((64, 1), 0.5 * i)) for i in range(1, 5)]
    with torch.no_grad():
        for w, s in values:
            mod.parametrizations.weight.original.copy_(w)
            mod.parametrizations.weight_scale.original.copy_(s)
            q, flat = mod._qweight(), mod._wscale_flat()
            assert torch.equal(q.float(), 2 * w) and torch.equal(flat, 2 * s.reshape(-1))


def test_awq_size_queries_answer_for_any_sizes():
    """In a child process: a division by a plan's zero tile count would end the whole process, not raise."""
    import subprocess
    import sys
    code = ("import itertools; from llmqrt_amd import _abi; L = _abi.lib(); v = (-1, 0, 1, 7, 8, 16, 31, 32, 33, 64, 65, 128, 300)\n"
            "for m, n, k in itertools.product(v, v, v):\n"
            "    L.llmq_awq_gemm_workspace_bytes(m, n, k)\n"
            "    for g in (-1, 0, 8, 32, 128): L.llmq_awq_gemm_partials_bytes(m, n, k, g)\n"
            "assert L.llmq_awq_gemm_workspace_bytes(1, 4608, 3584) > L.llmq_awq_gemm_partials_bytes(1, 4608, 3584, 128) > 0")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]


def test_queries_answer_for_the_largest_sizes():
    """Tile counts past 32 bits: sizes that no call takes need nothing, and a plan's division by a wrapped count would end the process."""
    import subprocess
    import sys
    code = ("import ctypes, itertools; from llmqrt_amd import _abi; L = _abi.lib(); c = ctypes.c_int()\n"
            "v = (1, 64, 70000, 2**24, 2**31 - 8, 2**31 - 1, 2**31, 2**40)\n"
            "for m, n, k in itertools.product(v, v, (64, 128, 2**22 - 16, 2**22, 2**31 - 32, 2**40)):\n"
            "    refused = max(m, n) >= 2**31 or k >= 2**22\n"
            "    for f in (0, 1): assert (L.llmq_gemm_planned_config(f, m, n, k) < 0) == refused\n"
            "    for q in ('gemm_w8a8', 'gemm_fp8', 'gemm', 'gemm_f16', 'gemm_fp8_quantized_output'):\n"
            "        assert getattr(L, f'llmq_{q}_workspace_bytes')(m, n, k) == 0 or not refused\n"
            "    if m > 2**24: continue  # the AWQ queries go over M in steps\n"
            "    L.llmq_awq_gemm_workspace_bytes(m, n, k)\n"
            "    for g in (32, 128):\n"
            "        L.llmq_awq_gemm_partials_bytes(m, n, k, g); L.llmq_awq_linear_partials_bytes(1, m, n, k, g, k, ctypes.byref(c))\n"
            "        L.llmq_awq_planned_config(1, m, n, k, g, k)\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]


def test_captured_calls_keep_no_shared_workspace(monkeypatch):
    """A capture neither uses a cached buffer, which a larger eager call would replace under the graph, nor leaves one."""
    from llmqrt_amd import _abi
    state = {"capturing": False}
    monkeypatch.setattr(torch.cuda, "current_device", lambda: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: type("S", (), {"cuda_stream": 7})())
    cache, cpu = _abi._Workspaces(), torch.device("cpu")
    assert cache.get(cpu, 0) is None
    eager = cache.get(cpu, 100)
    assert cache.get(cpu, 1 << 20) is eager and cache.get(cpu, (1 << 20) + 1) is not eager
    eager = cache.get(cpu, 1)
    state["capturing"] = True
    first, second = cache.get(cpu, 100), cache.get(cpu, 4 << 20)
    assert first is not eager and second is not eager and second is not first and second.numel() >= 4 << 20
    state["capturing"] = False
    assert cache.get(cpu, 100) is eager


def test_workspaces_are_bounded_and_given_back(monkeypatch):
    import llmqrt_amd
    from llmqrt_amd import _abi
    stream = {"id": 0}
    monkeypatch.setattr(torch.cuda, "current_device", lambda: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: type("S", (), {"cuda_stream": stream["id"]})())
    cache, cpu = _abi._Workspaces(), torch.device("cpu")
    monkeypatch.setattr(_abi, "workspaces", cache)
    monkeypatch.setattr(_abi._Workspaces, "_MAX_STREAMS", 4)
    for stream["id"] in range(9):
        assert cache.get(cpu, 8) is cache.get(cpu, 8) and len(cache._buf) <= 4
    llmqrt_amd.release_workspaces()
    assert not cache._buf


def test_native_library_of_another_torch_is_refused(monkeypatch):
    from llmqrt_amd import _native
    assert _native.host().torch_version == torch.__version__
    monkeypatch.setattr(torch, "__version__", "0.0.0")
    with pytest.raises(RuntimeError, match="built against torch"):
        _native._load()
