"""The streaming AWQ tile kernel (awq_stream.hip): every configuration at the edges of its tiles, stages, units and slices, forced through the
tuning hook, against fp64 sums; the bf16 form; workspaces."""
import pytest
import torch

from oracle import ref_math as R

pytestmark = pytest.mark.gpu


@pytest.fixture
def force():
    from llmqrt_amd import _abi
    L = _abi.lib()
    yield lambda cfg, splits: _abi.check(L.llmq_awq_force_plan(12 + cfg, splits, 0), "llmq_awq_force_plan")
    L.llmq_awq_force_plan(0, 0, 0)


def _problem(M, K, N, G, seed, xstride=0):
    from llmqrt_amd import workloads as W
    qw, qz, s = W.awq_weights(N, K, seed, group=G)
    x = W.activations(M, xstride or K, seed + 1, dtype=torch.float16, outliers=True)[:, :K]
    bias = torch.randn(N, generator=torch.Generator().manual_seed(seed)).half()
    return qw, qz, s, x, bias


def _reference(x, qw, qz, s, G, exact):
    """fp64 sums and the sums of absolute products; exact: the weights are (q - z) s, otherwise rounded to fp16 as the dequantizer does."""
    if exact:
        ones = torch.ones_like(s)
        w = R.awq_dequantize(qw, qz, ones, G).double() * s.double().repeat_interleave(G, 0)
    else:
        w = R.awq_dequantize(qw, qz, s, G).double()
    return x.double() @ w, x.double().abs() @ w.abs()


def _linear(x, qw, s, qz, G, bias=None):
    """llmq_awq_linear itself: the Python op refuses groups other than 32, 64, 128 and K, as the reference's does."""
    from llmqrt_amd import _abi
    L = _abi.lib()
    (M, K), N = x.shape, s.shape[1]
    need = L.llmq_awq_gemm_partials_bytes(M, N, K, G)
    out = torch.empty((M, N), dtype=x.dtype, device=x.device)
    tickets = torch.zeros(L.llmq_awq_workspace_ticket_bytes(), dtype=torch.uint8, device=x.device)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=x.device)
    _abi.check(L.llmq_awq_linear(x.data_ptr(), _abi.dtype_code(x.dtype), x.stride(0), qw.data_ptr(), s.data_ptr(), qz.data_ptr(), _abi.ptr(bias),
                                 out.data_ptr(), M, N, K, G, tickets.data_ptr(), ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream),
               "llmq_awq_linear")
    return out


# (M, K, N, G): one token, one row less and one more than a token tile and a slab, one stage, one unit, a unit and a half, fewer units than
# slices, column tiles that end inside (N % 256), channel counts that are no whole 16-byte pieces of packed words (N % 32), every kind of group:
# two per stage, one per stage, one across a stage and a half, one per unit, several units, the whole K; many splits
SHAPES = [(1, 64, 8, 64), (31, 128, 32, 128), (32, 192, 264, 32), (33, 192, 256, 96), (64, 256, 520, 128), (65, 640, 1056, 64),
          (127, 1024, 264, 1024), (128, 896, 1152, 128), (129, 384, 96, 384), (200, 768, 1000, 256), (300, 3584, 512, 128)]


@pytest.mark.parametrize("cfg", range(5))
@pytest.mark.parametrize("splits", [0, 1, 3, 24])
@pytest.mark.parametrize("M,K,N,G", SHAPES)
def test_every_configuration(cuda, force, cfg, splits, M, K, N, G):
    qw, qz, s, x, bias = _problem(M, K, N, G, 5 * M + N + K, K + 8 * (M % 3))
    with_bias = splits in (0, 3)
    exact = G % 128 == 0 and cfg <= 2  # the configurations of up to 64 tokens scale whole groups in fp32
    ref, mag = _reference(x, qw, qz, s, G, exact)
    # K fp32 additions of exact products (one rounding of a group's sum and one of its scaling more where whole groups are scaled), then the
    # rounding to fp16; with a bias another
    bound = (K + 2 * K // G) * 2.0 ** -24 * mag + 2.0 ** -11 * ref.abs() + 2.0 ** -24
    if with_bias:
        ref = ref + bias.double()
        bound = bound + 2.0 ** -11 * ref.abs()
    xd = torch.zeros((M, x.stride(0)), dtype=torch.float16)
    xd[:, :K] = x
    xd = xd.to(cuda)[:, :K]
    args = [t.to(cuda) for t in (qw, s, qz)]
    b = bias.to(cuda) if with_bias else None
    force(cfg, splits)
    out = _linear(xd, *args, G, b)
    err = (out.double().cpu() - ref).abs()
    assert bool((err <= bound).all()), (cfg, splits, M, K, N, G, float((err / bound).max()))
    if not with_bias:
        # The bound above holds for every element and is far from what sums of K terms lose: their errors add like a random walk, 2^-24 sqrt(K) of the size
        # of a partial sum.  Four times that moves an element across a rounding boundary with a chance of twice it over the fp16 spacing there.
        w = R.awq_dequantize(qw, qz, s, G).double()
        size = ((x.double() ** 2) @ (w ** 2) + ref ** 2).sqrt()
        spacing = torch.exp2(torch.floor(torch.log2(ref.abs().clamp(min=2.0 ** -14))) - 10)
        chance = (2 * 4 * 2.0 ** -24 * K ** 0.5 * size / spacing).clamp(max=1).sum().item()
        moved = int((out.cpu() != ref.half()).sum())
        assert moved <= chance + 4 * chance ** 0.5 + 2, (moved, chance, ref.numel())
    assert torch.equal(out, _linear(xd, *args, G, b)), "deterministic"
    # a bf16 model: the same op between x.half() and .bfloat16(), bit for bit
    xb = xd.bfloat16()
    assert torch.equal(_linear(xb, *args, G, b), _linear(xb.half(), *args, G, b).bfloat16())


@pytest.mark.parametrize("cfg", range(5))
def test_rows_do_not_leak_and_extremes(cuda, force, cfg):
    """A token row of infinities and NaN changes no other row; all-15 weights against zero points 0 and the reverse; fp16 overflow in the sum."""
    from llmqrt_amd.awq_kernels import awq_gemm_triton
    M, K, N, G = 70, 256, 288, 128
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(3)).half()
    s = (torch.rand(K // G, N, generator=torch.Generator().manual_seed(4)) * 0.02 + 0.001).half()
    force(cfg, 0)
    for qv, zv in ((15, 0), (0, 15)):
        qw, qz = R.awq_pack(torch.full((K, N), qv, dtype=torch.int32)), R.awq_pack(torch.full((K // G, N), zv, dtype=torch.int32))
        args = [t.to(cuda) for t in (qw, s, qz)]
        clean = awq_gemm_triton(x.to(cuda), *args, split_k_iters=8)
        ref, mag = _reference(x, qw, qz, s, G, cfg <= 2)
        assert bool(((clean.double().cpu() - ref).abs() <= K * 2.0 ** -23 * mag + 2.0 ** -11 * ref.abs() + 2.0 ** -24).all())
        bad = x.clone()
        bad[5, 17], bad[40, 200], bad[69, 3] = float("inf"), float("nan"), -float("inf")
        got = awq_gemm_triton(bad.to(cuda), *args, split_k_iters=8)
        keep = torch.ones(M, dtype=torch.bool)
        keep[[5, 40, 69]] = False
        assert torch.equal(got[keep.to(cuda)], clean[keep.to(cuda)])
        assert torch.isinf(got[5]).all() and torch.isnan(got[40]).all() and torch.isinf(got[69]).all()
        big = awq_gemm_triton((x * 0 + 60000).to(cuda), *args, split_k_iters=8)
        assert torch.isinf(big).all() and bool((big > 0).all()) == (qv == 15)


@pytest.mark.parametrize("M,K,N,G", [(24, 3584, 18944, 128), (64, 18944, 3584, 128), (40, 896, 896, 128), (9, 4864, 5248, 32), (200, 3584, 1152, 64),
                                     (777, 1024, 2048, 128), (28, 1536, 1000, 128)])
def test_plans_of_the_rules(cuda, M, K, N, G):
    """The plan that the rules pick, on both sides of the few-token kernel's range, through the module: fp16 and bf16, native and general path."""
    from llmqrt_amd.linear import WQLinear_GEMM
    qw, qz, s, x, bias = _problem(M, K, N, G, M + N)
    mod = WQLinear_GEMM(4, G, K, N, True, cuda)
    mod.qweight.copy_(qw); mod.qzeros.copy_(qz); mod.scales.copy_(s); mod.bias.copy_(bias)
    for dt in (torch.float16, torch.bfloat16):
        xd = x.to(dt).to(cuda)
        w = R.awq_dequantize(qw, qz, torch.ones_like(s), G).double() * s.double().repeat_interleave(G, 0)
        xf = xd.half().double().cpu()
        ref, mag = xf @ w, xf.abs() @ w.abs()
        y = mod(xd.view(1, M, K))[0]
        assert y.dtype == dt
        # a weight may be rounded to fp16 first (2^-11 of every product), the result to fp16 twice and to bf16
        tol = (K * 2.0 ** -24 + 2.0 ** -11) * mag + (2.0 ** -10 + (2.0 ** -8 if dt == torch.bfloat16 else 0)) * (ref.abs() + bias.double().abs()) + 2.0 ** -24
        assert bool(((y.double().cpu() - ref - bias.double()).abs() <= tol).all())
        pad = torch.zeros((M, K + 8), dtype=dt, device=cuda)
        pad[:, :K] = xd
        assert torch.equal(mod(pad[:, :K].unsqueeze(0))[0], y)  # strided rows: the general path


def test_workspace_rule(cuda):
    """A workspace of the query's size runs the plan; one that is enough for the kernels other than this one still runs, with fewer splits; a
    smaller one is refused before any launch, as it was."""
    from llmqrt_amd import _abi
    L = _abi.lib()
    M, K, N, G = 64, 18944, 3584, 128
    qw, qz, s, x, _ = (t.to(cuda) for t in _problem(M, K, N, G, 11))
    full = L.llmq_awq_gemm_partials_bytes(M, N, K, G)
    assert L.llmq_awq_gemm_workspace_bytes(M, N, K) >= full + L.llmq_awq_workspace_ticket_bytes()
    tickets = torch.zeros(L.llmq_awq_workspace_ticket_bytes(), dtype=torch.uint8, device=cuda)
    ws = torch.empty(full, dtype=torch.uint8, device=cuda)
    stream = torch.cuda.current_stream().cuda_stream

    def call(nbytes):
        out = torch.zeros((M, N), dtype=torch.float16, device=cuda)
        rc = L.llmq_awq_gemm_tickets(x.data_ptr(), _abi.F16, K, qw.data_ptr(), s.data_ptr(), qz.data_ptr(), None, out.data_ptr(), M, N, K, G,
                                     tickets.data_ptr(), ws.data_ptr(), nbytes, stream)
        return rc, out
    rc, out = call(full)
    assert rc == 0
    few = 4 * M * N * 4  # four splits of the few-token kernel
    rc, out4 = call(few)
    assert rc == 0 and ((out4.float() - out.float()).abs().max() <= 2e-3 * out.float().abs().max())
    rc, none = call(few // 4)
    assert rc == -4 and int(none.count_nonzero()) == 0


@pytest.mark.parametrize("M,K,N,G,dtype,most", [(777, 1024, 2048, 128, torch.float16, 1), (64, 18944, 3584, 128, torch.float16, 2), (12, 896, 1152, 32, torch.float16, 1),
                                                (12, 896, 1152, 32, torch.bfloat16, 2)])
def test_module_allocates_what_runs(cuda, M, K, N, G, dtype, most):
    """The output, and partial sums only where the kernel that runs splits K; arrival counters only for the kernel that counts (the 7B-class sizes
    above): a streaming call makes none."""
    from llmqrt_amd._native import host
    from llmqrt_amd.linear import WQLinear_GEMM
    qw, qz, s, x, _ = _problem(M, K, N, G, M + N)
    mod = WQLinear_GEMM(4, G, K, N, False, cuda)
    mod.qweight.copy_(qw); mod.qzeros.copy_(qz); mod.scales.copy_(s)
    xd = x.to(dtype).to(cuda).view(1, M, K)
    ref = mod(xd)
    torch.cuda.synchronize()
    host().release_tickets()
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    y = mod(xd)
    assert torch.cuda.memory_stats()["allocation.all.allocated"] - before == most
    assert torch.equal(y, ref)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_exact_workspace_without_counters(cuda, dtype):
    """llmq_awq_linear with the bytes that its query names and no counters gives what it gives with more of both; with no workspace at all it runs
    without a split or refuses, as the kernels before need one; the few-token kernel refuses a split without counters."""
    import ctypes
    from llmqrt_amd import _abi
    L = _abi.lib()
    stream = torch.cuda.current_stream().cuda_stream
    tickets = torch.zeros(L.llmq_awq_workspace_ticket_bytes(), dtype=torch.uint8, device=cuda)

    def call(M, K, N, G, tick, ws, nbytes):
        qw, qz, s, x, _ = (t.to(cuda) for t in _problem(M, K, N, G, M))
        out = torch.zeros((M, N), dtype=dtype, device=cuda)
        rc = L.llmq_awq_linear(x.to(dtype).data_ptr(), _abi.dtype_code(dtype), K, qw.data_ptr(), s.data_ptr(), qz.data_ptr(), None, out.data_ptr(), M, N, K, G,
                               _abi.ptr(tick), _abi.ptr(ws), nbytes, stream)
        return rc, out
    flag = ctypes.c_int(0)
    for M, K, N, G in ((64, 18944, 3584, 128), (200, 3584, 1152, 64), (130, 1024, 520, 128)):
        need = L.llmq_awq_linear_partials_bytes(_abi.dtype_code(dtype), M, N, K, G, K, ctypes.byref(flag))
        assert flag.value == 0
        guard = torch.full((need + 256,), 0x5A, dtype=torch.uint8, device=cuda)
        rc, exact = call(M, K, N, G, None, guard, need)
        big = torch.empty(max(need, L.llmq_awq_gemm_partials_bytes(M, N, K, G), 16), dtype=torch.uint8, device=cuda)
        rc2, ref = call(M, K, N, G, tickets, big, big.numel())
        assert rc == rc2 == 0 and torch.equal(exact, ref) and bool((guard[need:] == 0x5A).all())
        rc, _ = call(M, K, N, G, None, None, 0)
        assert rc == (-4 if L.llmq_awq_gemm_partials_bytes(M, N, K, G) else 0)
    need = L.llmq_awq_linear_partials_bytes(_abi.dtype_code(dtype), 4, 3584, 3584, 128, 3584, ctypes.byref(flag))
    assert need and flag.value == 1
    rc, none = call(4, 3584, 3584, 128, None, torch.empty(need, dtype=torch.uint8, device=cuda), need)
    assert rc == -4 and int(none.count_nonzero()) == 0
