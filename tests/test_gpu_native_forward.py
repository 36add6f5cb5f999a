"""The native forward passes of the modules (csrc/host_ops.cpp) against the general Python path of the same module."""
import pytest
import torch

pytestmark = pytest.mark.gpu

K, N = 1024, 544


def _modules(dtype, bias):
    from llmqrt_amd.linear import (FP8DynamicLinear, FP8StaticLinear, SqW8A8BBF16OBF16PerChannel,
                                   SqW8A8BBF16OBF16PerTensor, WQLinear_GEMM)
    g = torch.Generator(device="cuda").manual_seed(5)
    lin = torch.nn.Linear(K, N, bias=bias, device="cuda")
    lin.weight.data = 0.02 * torch.randn(N, K, device="cuda", generator=g)
    if bias:
        lin.bias.data = torch.randn(N, device="cuda", generator=g)
    mods = {"sq": SqW8A8BBF16OBF16PerTensor.from_linear(lin, 8, 0, False, dtype=dtype),
            "sq_channel": SqW8A8BBF16OBF16PerChannel.from_linear(lin, 8, 0, False, dtype=dtype),
            "fp8": FP8DynamicLinear.from_linear(lin, init_only=False, dtype=dtype, per_tensor=True)}
    for name, quantized in (("static", False), ("static_out", True)):
        m = FP8StaticLinear.from_linear(lin, init_only=False, dtype=dtype, quantize_output=quantized)
        m.input_scale.data.fill_(0.15)
        m.output_scale.data.fill_(0.05)
        mods[name] = m
    if dtype == torch.bfloat16:
        mods["fp8_token"] = FP8DynamicLinear.from_linear(lin, init_only=False, dtype=dtype, per_tensor=False)
    w = lin.weight.t().reshape(K // 128, 128, N)
    s = ((w.amax(1) - w.amin(1)) / 15).clamp(min=1e-5).half()
    z = (-w.amin(1) / s.float()).round().clamp(0, 15)
    mods["awq"] = WQLinear_GEMM.from_linear(lin, 4, 128, scales=s, zeros=z)
    return mods


# 1 - 5 tokens: one-launch linears; 70 and 300: tile kernels, AWQ streaming; 450: AWQ dequantize + GEMM
@pytest.mark.parametrize("M", [1, 4, 5, 70, 300, 450])
@pytest.mark.parametrize("dtype,bias", [(torch.bfloat16, True), (torch.float16, False)])
def test_native_forward_equals_general_path(cuda, M, dtype, bias):
    x = torch.randn(M, 1, K, device=cuda, generator=torch.Generator(device="cuda").manual_seed(M)).to(dtype)
    strided = torch.zeros(M, 1, K + 8, dtype=dtype, device=cuda)
    strided[..., :K] = x
    from llmqrt_amd.linear.linear_awq import dequant_matmul_token_threshold
    assert 300 < dequant_matmul_token_threshold(K, N) <= 450
    for name, mod in _modules(dtype, bias).items():
        y, ref = mod(x), mod._forward_general(x)
        assert y.shape == (M, 1, N) and y.dtype == ref.dtype, name
        assert torch.equal(y, ref), name
        assert torch.equal(mod(strided[..., :K]), ref), name  # not contiguous: the general path from forward()


@pytest.mark.parametrize("fp8", [False, True])
def test_native_norm_and_prequantized(cuda, fp8):
    from llmqrt_amd.norm import RMSNorm, rmsnorm, rmsnorm_per_token_quantize, rmsnorm_quantize_activation_per_token_absmax
    mods = _modules(torch.bfloat16, True)
    mod = mods["fp8_token" if fp8 else "sq_channel"]
    g = torch.Generator(device="cuda").manual_seed(9)
    x = torch.randn(2, 37, K, device=cuda, generator=g).bfloat16()
    norm = RMSNorm((1 + 0.1 * torch.randn(K, device=cuda, generator=g)).bfloat16(), 1e-6)
    assert torch.equal(norm(x), rmsnorm(x, norm.weight, 1e-6))
    q, s = norm.forward_quantized(x, fp8=fp8)
    if fp8:
        q2, s2 = rmsnorm_per_token_quantize(x, norm.weight, 1e-6)
        y, ref = mod.forward_quantized(q, s), mod._forward_quantized_general(q, s)
    else:
        q2, s2 = rmsnorm_quantize_activation_per_token_absmax(x, norm.weight, 1e-6, torch.float32)
        y, ref = mod.forward_quantized(q, s, x.dtype), mod._forward_quantized_general(q, s, x.dtype)
    assert torch.equal(q.view(torch.uint8), q2.view(torch.uint8)) and torch.equal(s, s2)
    assert q.shape == x.shape and s.shape == (2, 37, 1) and y.shape == (2, 37, N) and torch.equal(y, ref)


def test_native_awq_counters_by_stream(cuda):
    """K splits that end in arrival counters: calls overlapping on two streams, and a captured call replayed beside them."""
    mod = _modules(torch.bfloat16, False)["awq"]
    g = torch.Generator(device="cuda").manual_seed(3)
    xs = [torch.randn(4, K, device=cuda, generator=g).bfloat16() for _ in range(2)]
    refs = [mod._forward_general(x) for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = mod(xs[0])
    outs = [[], []]
    for _ in range(20):
        for i, st in enumerate(streams):
            with torch.cuda.stream(st):
                outs[i].append(mod(xs[i]))
        graph.replay()
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(y, refs[i]) for y in outs[i])
    assert torch.equal(captured, refs[0])


def test_captured_awq_call_owns_its_counters(cuda):
    """A graph captured on a stream that already has counters keeps none of them: they may go, or count for eager calls."""
    from llmqrt_amd._native import host
    mod = _modules(torch.bfloat16, False)["awq"]
    x = torch.randn(4, K, device=cuda, generator=torch.Generator(device="cuda").manual_seed(3)).bfloat16()
    st, other = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(st):
        ref = mod(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        captured = mod(x)
    outs = []
    for _ in range(10):
        with torch.cuda.stream(st):
            outs.append(mod(x))
        with torch.cuda.stream(other):
            graph.replay()
    torch.cuda.synchronize()
    host().release_tickets()
    outs.append(mod(x))
    with torch.cuda.stream(other):
        graph.replay()
    torch.cuda.synchronize()
    assert all(torch.equal(y, ref) for y in outs) and torch.equal(captured, ref)


def test_replica_forward_equals_module(cuda):
    """A DataParallel replica: its parameters are plain attributes, so the general path serves the fp8 modules."""
    x = torch.randn(5, K, device=cuda, generator=torch.Generator(device="cuda").manual_seed(1)).bfloat16()
    for name, mod in _modules(torch.bfloat16, True).items():
        rep = mod._replicate_for_data_parallel()
        for key, p in mod._parameters.items():
            setattr(rep, key, p.detach())
        assert torch.equal(rep(x), mod._forward_general(x)), name


@pytest.mark.parametrize("M", [3, 70])
@pytest.mark.parametrize("cast", [torch.bfloat16, torch.float16])
def test_fp8_modules_cast_to_16_bits(cuda, M, cast):
    """module.to(16-bit dtype) casts the scales too: activation scale x weight scale is then torch's product of the two."""
    from llmqrt_amd.quantize import per_tensor_quantize, static_per_tensor_quantize
    from llmqrt_amd.sq_fp8_kernels import cutlass_f8f8bf16_tensorwise_sm89
    x = torch.randn(M, K, device=cuda, generator=torch.Generator(device="cuda").manual_seed(M)).to(cast)
    mods = _modules(cast, True)
    for name in ("fp8", "static"):
        mod = mods[name].to(cast)
        assert mod.weight_scale.dtype == cast
        if name == "fp8":
            q, s = per_tensor_quantize(x)
        else:
            q, s = static_per_tensor_quantize(x, mod.input_scale), mod.input_scale
        ref = cutlass_f8f8bf16_tensorwise_sm89(q, mod._qweight_t(), mod.bias, mod.weight_scale * s, 1.0,
                                               "bfloat16" if cast == torch.bfloat16 else "float16")
        assert torch.equal(mod(x), ref), name


def test_static_input_scale_off_the_gpu_is_refused(cuda):
    """A one-dimensional host scale: torch refuses the product with the weight's scale, and so does the module."""
    mod = _modules(torch.bfloat16, True)["static"]
    mod.input_scale.data = mod.input_scale.data.cpu()
    x = torch.randn(3, K, device=cuda).bfloat16()
    with pytest.raises(RuntimeError):
        mod(x)
    from llmqrt_amd.quantize import per_tensor_quantize_with_alpha
    with pytest.raises(RuntimeError, match="weight scale"):
        per_tensor_quantize_with_alpha(x, torch.ones(1), True)


def _allocations():
    return torch.cuda.memory_stats()["allocation.all.allocated"]


@pytest.mark.parametrize("form", ["module", "op"])
def test_capture_zeroes_counters_once(cuda, form):
    """A captured AWQ call with a K split allocates its output and partial sums; the counters are one set per capture and
    stream.  Replays beside eager work, with a second stream inside the graph and the pool released in between, stay right."""
    from llmqrt_amd._native import host
    from llmqrt_amd.awq_kernels import awq_gemm_triton
    mod = _modules(torch.bfloat16, False)["awq"]
    g = torch.Generator(device="cuda").manual_seed(8)
    xs = [torch.randn(4, K, device=cuda, generator=g).half() for _ in range(4)]
    call = mod if form == "module" else lambda x: awq_gemm_triton(x, mod.qweight, mod.scales, mod.qzeros, 8)
    refs = [call(x) for x in xs]
    torch.cuda.synchronize()
    st, side = torch.cuda.Stream(), torch.cuda.Stream()
    graphs, counts = [], []
    for calls in (1, 3):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=st):
            before = _allocations()
            ys = [call(xs[i]) for i in range(calls)]
            counts.append(_allocations() - before)
            ptr = host().awq_counters(xs[0]).data_ptr()
            assert host().awq_counters(xs[0]).data_ptr() == ptr
            side.wait_stream(st)
            with torch.cuda.stream(side):
                ys.append(call(xs[3]))
                assert host().awq_counters(xs[0]).data_ptr() != ptr
            st.wait_stream(side)
        graphs.append((graph, ys, refs[:calls] + refs[3:]))
    assert counts[1] - counts[0] == 2 * 2  # output and partial sums of two more calls
    for turn in range(5):
        for graph, ys, want in graphs:
            for y in ys:
                y.zero_()
            graph.replay()
            with torch.cuda.stream(st):
                eager = call(xs[turn % 4])
            torch.cuda.synchronize()
            assert torch.equal(eager, refs[turn % 4])
            assert all(torch.equal(y, r) for y, r in zip(ys, want))
        if turn == 2:
            host().release_tickets()


def test_more_streams_than_counter_sets(cuda):
    """256 streams keep a counter set; a call on one more zeroes a set of its own, and gives the same result."""
    import ctypes
    import llmqrt_amd
    from llmqrt_amd._native import host
    hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))
    mod = _modules(torch.bfloat16, False)["awq"]
    x = torch.randn(4, K, device=cuda, generator=torch.Generator(device="cuda").manual_seed(2)).bfloat16()
    ref = mod(x)
    torch.cuda.synchronize()
    llmqrt_amd.release_workspaces()
    kept = []
    for i in range(258):
        ptr = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(ptr)) == 0
        with torch.cuda.stream(torch.cuda.ExternalStream(ptr.value)):
            host().awq_counters(x)
            before = _allocations()
            host().awq_counters(x)
            kept.append(_allocations() == before)
            y = mod(x) if i in (0, 255, 256, 257) else None
        torch.cuda.synchronize()
        assert y is None or torch.equal(y, ref), i
    assert kept == [True] * 256 + [False] * 2
    llmqrt_amd.release_workspaces()


@pytest.mark.parametrize("M", [1, 5, 70, 300])
@pytest.mark.parametrize("dtype,bias", [(torch.bfloat16, True), (torch.float16, False)])
def test_contiguous_rows_take_the_native_call(cuda, M, dtype, bias, monkeypatch):
    """What the comparisons of this file rest on: contiguous activations never reach the general path, strided ones do."""
    from llmqrt_amd import norm as norm_module

    class General(Exception):
        pass

    def general(*args, **kwargs):
        raise General

    wide = torch.randn(M, 1, K + 8, device=cuda, generator=torch.Generator(device="cuda").manual_seed(M)).to(dtype)
    x, strided = wide[..., :K].contiguous(), wide[..., :K]
    norm = norm_module.RMSNorm(torch.ones(K, device=cuda, dtype=dtype))
    mods = _modules(dtype, bias)
    for name in ("rmsnorm", "rmsnorm_per_token_quantize", "rmsnorm_quantize_activation_per_token_absmax"):
        monkeypatch.setattr(norm_module, name, general)
    calls = [norm, norm.forward_quantized, lambda t: norm.forward_quantized(t, fp8=True)]
    for mod in mods.values():
        monkeypatch.setattr(mod, "_forward_general", general)
        calls.append(mod)
    for call in calls:
        call(x)
        if M > 1:
            with pytest.raises(General):
                call(strided)
    quantized = {"sq_channel": (torch.int8, (dtype,)), "fp8_token": (torch.float8_e4m3fn, ())}
    for name, (qdtype, more) in quantized.items():
        if name in mods:
            monkeypatch.setattr(mods[name], "_forward_quantized_general", general)
            mods[name].forward_quantized(x.to(qdtype), torch.ones(M, 1, 1, device=cuda), *more)


def test_native_forward_from_threads(cuda):
    """Four threads on a stream each share the modules and the counter pool while a fifth gives the pool back."""
    import threading
    from llmqrt_amd._native import host
    mods = list(_modules(torch.bfloat16, True).items())
    g = torch.Generator(device="cuda").manual_seed(6)
    xs = [torch.randn(m, 1, K, device=cuda, generator=g).bfloat16() for m in (1, 4, 5, 70)]
    refs = [[mod._forward_general(x) for _, mod in mods] for x in xs]
    torch.cuda.synchronize()
    wrong, done = [], threading.Event()

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                ys = [mod(xs[i]) for _, mod in mods]
                torch.cuda.current_stream().synchronize()
                wrong.extend((i, name) for (name, _), y, ref in zip(mods, ys, refs[i]) if not torch.equal(y, ref))

    def release():
        while not done.wait(0.002):
            host().release_tickets()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    releaser = threading.Thread(target=release)
    releaser.start()
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    done.set()
    releaser.join(10)
    assert not wrong and not any(t.is_alive() for t in threads + [releaser])


# 16 x 896 x 4864 and 14 x 416 x 4096 run in one launch from a program's loop and in two inside a graph, where no host waits for the second
@pytest.mark.parametrize("M,n,k", [(16, 896, 4864), (14, 416, 4096), (16, 3584, 2304)])
@pytest.mark.parametrize("name", ["sq", "fp8", "sq_channel", "fp8_token", "static", "static_out"])
def test_captured_forward_follows_the_gpu(cuda, M, n, k, name):
    """int8 results are the eager ones bit for bit; fp8 sums may be added in another order (twice K 2^-24 of the sum of absolute products, a step of the output type).
    Every replay equals the first, with eager calls between them."""
    from llmqrt_amd.linear import FP8DynamicLinear, FP8StaticLinear, SqW8A8BBF16OBF16PerChannel, SqW8A8BBF16OBF16PerTensor
    g = torch.Generator(device="cuda").manual_seed(n)
    lin = torch.nn.Linear(k, n, bias=False, device="cuda")
    lin.weight.data = 0.02 * torch.randn(n, k, device="cuda", generator=g)
    if name.startswith("sq"):
        mod = (SqW8A8BBF16OBF16PerTensor if name == "sq" else SqW8A8BBF16OBF16PerChannel).from_linear(lin, 8, 0, False, dtype=torch.bfloat16)
    elif name.startswith("static"):
        mod = FP8StaticLinear.from_linear(lin, init_only=False, dtype=torch.bfloat16, quantize_output=name == "static_out")
        mod.input_scale.data.fill_(0.02)
        mod.output_scale.data.fill_(0.02)
    else:
        mod = FP8DynamicLinear.from_linear(lin, init_only=False, dtype=torch.bfloat16, per_tensor=name == "fp8")
    x = torch.randn(M, 1, k, device=cuda, generator=g).bfloat16()
    eager = mod(x)
    st = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        before = _allocations()
        y = mod(x)
        made = _allocations() - before
    if name in ("sq", "fp8") and n < 1024:
        assert made == 2  # the output, and the codes of a separate quantizer
    graph.replay()
    torch.cuda.synchronize()
    first = y.clone()
    if name.startswith("sq"):
        assert torch.equal(first, eager)
    else:
        mag = x.double().abs() @ (mod._qweight().double() * mod.weight_scale.double().reshape(-1, 1)).abs().t()
        tol = (2 * k * 2.0 ** -24 + 2.0 ** -12) * mag + 2.0 ** -8 * eager.double().abs() + (eager.double().abs() / 8 + 0.02 * 2.0 ** -9 if name == "static_out" else 0)
        assert bool(((first.double() - eager.double()).abs() <= tol).all())
    for _ in range(3):
        y.zero_()
        graph.replay()
        again = mod(x)
        torch.cuda.synchronize()
        assert torch.equal(y, first) and torch.equal(again, eager)


def _route_modules(dtype):
    """(name, module, activations) of calls that run the kernels of few tokens and short prompts: the row-streaming GEMM with one group of channels a block, with
    several and in three token tiles, the streaming AWQ kernel with a K split and without, for groups of 128 and 32."""
    import ctypes
    from llmqrt_amd import _abi
    from llmqrt_amd.linear import FP8DynamicLinear, SqW8A8BBF16OBF16PerChannel, WQLinear_GEMM
    L = _abi.lib()
    g = torch.Generator(device="cuda").manual_seed(12)
    calls = []
    for fp8, M, n, k in ((False, 24, 1536, 2048), (True, 24, 1536, 2048), (False, 9, 16640, 1168), (True, 9, 16640, 8192), (True, 40, 2304, 2048)):
        assert 110 <= L.llmq_gemm_planned_config(int(fp8), M, n, k) <= 123
        lin = torch.nn.Linear(k, n, bias=False, device="cuda")
        lin.weight.data = 0.02 * torch.randn(n, k, device="cuda", generator=g)
        mod = FP8DynamicLinear.from_linear(lin, init_only=False, dtype=torch.bfloat16, per_tensor=False) if fp8 else \
            SqW8A8BBF16OBF16PerChannel.from_linear(lin, 8, 0, False, dtype=torch.bfloat16)
        calls.append((f"rows {M} x {n} x {k} {fp8}", mod, [torch.randn(M, k, device="cuda", generator=g).bfloat16() for _ in range(2)]))
    for M, n, k, group in ((64, 1024, 4096, 32), (48, 384, 2048, 64), (777, 2048, 1024, 128), (40, 896, 896, 128)):
        need = ctypes.c_int(0)
        assert L.llmq_awq_planned_config(_abi.dtype_code(dtype), M, n, k, group, k) >= 12
        split = L.llmq_awq_linear_partials_bytes(_abi.dtype_code(dtype), M, n, k, group, k, ctypes.byref(need)) > 0
        mod = WQLinear_GEMM(4, group, k, n, False, "cuda")
        mod.qweight.random_(generator=g)
        mod.qzeros.random_(generator=g)
        mod.scales.uniform_(0.001, 0.01, generator=g)
        calls.append((f"stream {M} x {n} x {k} {group} split {split}", mod, [torch.randn(M, k, device="cuda", generator=g).to(dtype) for _ in range(2)]))
    assert {name.endswith("split True") for name, _, _ in calls if name.startswith("stream")} == {True, False}
    return calls


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_streaming_kernels_captured_and_on_two_streams(cuda, dtype):
    """Captured calls replayed beside eager ones on two streams: every result is the one of a lone call, bit for bit."""
    calls = _route_modules(dtype)
    refs = [[mod(x) for x in xs] for _, mod, xs in calls]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=streams[0]):
        captured = [mod(xs[1]) for _, mod, xs in calls]
    for _ in range(4):
        for y in captured:
            y.zero_()
        torch.cuda.synchronize()
        outs = [[], []]
        for i, (_, mod, xs) in enumerate(calls):
            for j, st in enumerate(streams):
                with torch.cuda.stream(st):
                    outs[j].append(mod(xs[j]))
        with torch.cuda.stream(streams[1]):
            graph.replay()
        torch.cuda.synchronize()
        for i, (name, _, _) in enumerate(calls):
            assert torch.equal(outs[0][i], refs[i][0]) and torch.equal(outs[1][i], refs[i][1]), name
            assert torch.equal(captured[i], refs[i][1]), name


def test_streaming_kernels_from_threads(cuda):
    """Four threads on a stream each, each its own plans and scratch."""
    import threading
    calls = _route_modules(torch.bfloat16)
    refs = [[mod(x) for x in xs] for _, mod, xs in calls]
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(5):
                ys = [mod(xs[i % 2]) for _, mod, xs in calls]
                torch.cuda.current_stream().synchronize()
                wrong.extend((i, name) for (name, _, _), y, ref in zip(calls, ys, refs) if not torch.equal(y, ref[i % 2]))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not wrong and not any(t.is_alive() for t in threads)
