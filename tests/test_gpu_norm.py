"""GPU parity: RMSNorm and RMSNorm fused with the per-token quantizers vs the CPU oracle.

The reciprocal RMS depends on the fp32 summation order, so it is compared within a few fp32 ulps; every
other output is compared BIT-EXACTLY against the oracle evaluated with the kernel's own reciprocal RMS,
and end to end against the oracle's own within one rounding step on a vanishing fraction of elements."""
import pytest
import torch

from oracle import ref_math as R

pytestmark = pytest.mark.gpu

INV_RTOL = 5e-7  # ~4 ulp of fp32: summation order + one sqrt + one division
# (258, 896) .. (257, 520) take the wavefront-per-row kernels (256 rows or more of at most 1024 elements); then both sides of the row counts
# and row lengths at which the block of a row changes: 257-512 chunks (512 threads below 256 rows, 256 below 768, 128), 513-1024, 1025-2560
# (512 threads up to 256 rows, 256)
SHAPES = [(1, 896), (16, 896), (7, 3584), (128, 3584), (33, 18944), (3, 8), (5, 24576), (2, 40960),
          (258, 896), (1027, 1024), (300, 8), (257, 520), (300, 3584), (257, 2056), (256, 4096),
          (255, 4096), (767, 2056), (768, 4096), (9, 4104), (300, 8192), (256, 8200), (257, 8200), (3, 20480)]


def _inputs(M, K, dtype, seed):
    from llmqrt_amd import workloads as W
    x = W.activations(M, K, seed, dtype=dtype)
    if M > 2:
        x[2] = 0  # all-zero row: inv = 1/sqrt(eps), y = 0, quantizer floor scale
    g = torch.Generator().manual_seed(seed + 1)
    w = (1.0 + 0.2 * torch.randn(K, generator=g)).to(dtype)
    return x, w


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K", SHAPES)
def test_rmsnorm(cuda, M, K, dtype):
    from llmqrt_amd.norm import rmsnorm
    x, w = _inputs(M, K, dtype, 5 * M + K)
    eps = 1e-6
    inv = torch.empty(M, dtype=torch.float32, device=cuda)
    y = rmsnorm(x.to(cuda), w.to(cuda), eps, _inv_dump=inv)
    y_ref, inv_ref = R.rmsnorm(x, w, eps)
    assert y.dtype == dtype and y.shape == x.shape
    assert torch.allclose(inv.cpu(), inv_ref.view(-1), rtol=INV_RTOL, atol=0)
    assert torch.equal(y.cpu().view(torch.int16), R.rmsnorm_given_inv(x, w, inv.cpu()).view(torch.int16))
    # end to end: a different last bit of inv can move x * inv across a rounding boundary, rarely; one step
    # of the normalised value (up to 2^-7 relative for bf16) then passes through the product with weight
    diff = (y.cpu().float() - y_ref.float()).abs()
    ulp = 2.0 ** (-6 if dtype == torch.bfloat16 else -9)
    assert (diff <= ulp * y_ref.float().abs() + 1e-30).all()
    assert (diff > 0).float().mean() < 2e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K", SHAPES)
def test_rmsnorm_int8_fused(cuda, M, K, dtype):
    from llmqrt_amd.norm import rmsnorm_quantize_activation_per_token_absmax as fused
    x, w = _inputs(M, K, dtype, 7 * M + K)
    eps = 1e-6
    inv = torch.empty(M, dtype=torch.float32, device=cuda)
    q, s, y = fused(x.to(cuda), w.to(cuda), eps, return_normed=True, _inv_dump=inv)
    y_ref = R.rmsnorm_given_inv(x, w, inv.cpu())
    q_ref, s_ref = R.quantize_activation_per_token_absmax(y_ref)
    assert torch.allclose(inv.cpu(), R.rmsnorm(x, w, eps)[1].view(-1), rtol=INV_RTOL, atol=0)
    assert torch.equal(y.cpu().view(torch.int16), y_ref.view(torch.int16))
    assert s.dtype == dtype and torch.equal(s.cpu().view(torch.int16), s_ref.view(torch.int16))
    assert torch.equal(q.cpu(), q_ref)
    # without the normalised output, with fp32 scales: same codes
    q2, s2 = fused(x.to(cuda), w.to(cuda), eps, scale_dtype=torch.float32)
    assert torch.equal(q2.cpu(), q_ref) and torch.equal(s2.cpu(), s_ref.float())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K", SHAPES)
def test_rmsnorm_fp8_fused(cuda, M, K, dtype):
    from llmqrt_amd.norm import rmsnorm_per_token_quantize as fused
    x, w = _inputs(M, K, dtype, 9 * M + K)
    eps = 1e-5
    inv = torch.empty(M, dtype=torch.float32, device=cuda)
    q, s, y = fused(x.to(cuda), w.to(cuda), eps, return_normed=True, _inv_dump=inv)
    y_ref = R.rmsnorm_given_inv(x, w, inv.cpu())
    q_ref, s_ref = R.fp8_per_token_quantize(y_ref)
    assert torch.equal(y.cpu().view(torch.int16), y_ref.view(torch.int16))
    assert torch.equal(s.cpu(), s_ref)
    assert torch.equal(q.cpu().view(torch.uint8), q_ref.view(torch.uint8))


@pytest.mark.parametrize("M,K", [(7, 3584), (300, 3584), (768, 2056), (300, 1024), (9, 4104), (9, 8200), (257, 8200), (3, 24576)])
def test_a_nan_stays_in_its_row(cuda, M, K):
    """One NaN makes its row's mean NaN: normalised row and scale are NaN, int8 codes 0, fp8 codes NaN; the other rows keep their bits."""
    from llmqrt_amd.norm import rmsnorm_per_token_quantize, rmsnorm_quantize_activation_per_token_absmax
    x, w = _inputs(M, K, torch.bfloat16, M * K)
    bad = x.clone()
    bad[1, K - 1] = float("nan")
    rest = [m for m in range(M) if m != 1]
    for fused in (rmsnorm_quantize_activation_per_token_absmax, rmsnorm_per_token_quantize):
        q0, s0, y0 = [t.cpu() for t in fused(x.to(cuda), w.to(cuda), 1e-6, return_normed=True)]
        q, s, y = [t.cpu() for t in fused(bad.to(cuda), w.to(cuda), 1e-6, return_normed=True)]
        assert y[1].isnan().all() and s[1].isnan().all()
        assert bool((q[1] == 0).all()) if q.dtype == torch.int8 else q[1].float().isnan().all()
        for a, b in ((q, q0), (s, s0), (y, y0)):
            assert torch.equal(a[rest].contiguous().view(torch.uint8), b[rest].contiguous().view(torch.uint8))


def _mean_square_in_order(x, M):
    """mean(x^2) in the kernels' order of fp32 additions for a problem of M rows (the square of a 16-bit float is exact in fp32, so an FMA
    adds like a plain addition): LANES running sums over the 16-byte chunks t, t + LANES, .., a butterfly over each 64 of them, the 64s in
    order."""
    rows, K = x.shape
    chunks = K // 8
    lanes = 64 if chunks <= 128 and M >= 256 else 128 if 256 < chunks <= 512 and M >= 256 else 256
    per_lane = -(-chunks // lanes)
    sq = torch.zeros(rows, per_lane * lanes, 8)
    sq[:, :chunks] = x.float().square().view(rows, chunks, 8)
    sq = sq.view(rows, per_lane, lanes, 8)
    acc = torch.zeros(rows, lanes)
    for c in range(per_lane):
        for e in range(8):
            acc = acc + sq[:, c, :, e]
    acc = acc.view(rows, lanes // 64, 64)
    for o in (32, 16, 8, 4, 2, 1):
        acc = acc + acc[..., torch.arange(64) ^ o]
    total = acc[:, 0, 0]
    for w in range(1, lanes // 64):
        total = total + acc[:, w, 0]
    return total / float(K)


# both sides of every row count at which the block of a row changes, every row length class; K is a power of two, so the mean is exact
@pytest.mark.parametrize("M,K", [(8, 1024), (300, 1024), (8, 2048), (300, 2048), (1, 4096), (255, 4096), (256, 4096), (399, 4096), (400, 4096),
                                 (767, 4096), (768, 4096), (6143, 4096), (6144, 4096), (9, 8192), (300, 8192), (3, 16384), (256, 16384),
                                 (257, 16384), (1024, 16384), (1025, 16384), (3, 32768)])
def test_order_of_the_sum_of_squares(cuda, M, K):
    """The bits of the sum follow from the size of the problem, whatever block adds it up.  The rows are permutations of one row, and eps takes
    all but a thousandth of its mean square away: one last bit of the sum (6e-8 of it) moves the result by 3e-5, a few last bits of the root
    and the reciprocal by 5e-7."""
    from llmqrt_amd.norm import rmsnorm
    g = torch.Generator().manual_seed(M + K)
    base = torch.randn(K, generator=g).bfloat16()
    rows = min(M, 64)
    x = torch.stack([base[torch.randperm(K, generator=g)] for _ in range(rows)]).repeat(-(-M // rows), 1)[:M].contiguous()
    mean = _mean_square_in_order(x[:rows], M)
    eps = torch.tensor(-0.999 * float(base.double().square().mean()), dtype=torch.float32)
    inv = torch.empty(M, dtype=torch.float32, device=cuda)
    rmsnorm(x.to(cuda), torch.ones(K, dtype=torch.bfloat16, device=cuda), float(eps), _inv_dump=inv)
    want = (1.0 / torch.sqrt((mean + eps).double())).repeat(-(-M // rows))[:M]
    assert ((inv.cpu().double() - want).abs() <= 1e-6 * want).all()


def test_strided_rows_and_3d(cuda):
    from llmqrt_amd.norm import RMSNorm
    x = torch.randn(2, 5, 1024, generator=torch.Generator().manual_seed(3)).bfloat16()
    w = torch.ones(512, dtype=torch.bfloat16)
    xs = x[..., :512]  # row stride 1024
    m = RMSNorm(w.to(cuda), 1e-6)
    y = m(xs.to(cuda))
    y_ref, _ = R.rmsnorm(xs, w, 1e-6)
    assert y.shape == (2, 5, 512)
    assert (y.cpu().float() - y_ref.float()).abs().max() <= 2.0 ** -7 * y_ref.float().abs().max()
    q, s = m.forward_quantized(xs.to(cuda))
    assert q.shape == (2, 5, 512) and s.shape == (2, 5, 1) and s.dtype == torch.float32
    assert m(torch.empty(0, 512, dtype=torch.bfloat16, device=cuda)).shape == (0, 512)


def test_norm_then_linear_matches_unfused(cuda):
    """The fused norm+quant feeding the W8A8 Linear gives exactly what norm -> Linear.forward gives."""
    from llmqrt_amd import workloads as W
    from llmqrt_amd.linear import SqW8A8BBF16OBF16PerChannel
    from llmqrt_amd.norm import RMSNorm
    K, N, M = 896, 4864, 16
    x = W.activations(M, K, 77, dtype=torch.bfloat16).to(cuda)
    norm = RMSNorm(torch.ones(K, dtype=torch.bfloat16, device=cuda) * 1.5, 1e-6)
    lin = SqW8A8BBF16OBF16PerChannel(8, 0, K, N, True, dev=cuda, dtype=torch.bfloat16)
    qw, ws = W.int8_weights(N, K, 78)
    lin.qweight.copy_(qw.to(cuda)); lin.weight_scale.copy_(ws.to(cuda))
    unfused = lin(norm(x))
    q, s = norm.forward_quantized(x)
    fused = lin.forward_quantized(q, s, torch.bfloat16)
    assert torch.equal(unfused, fused)
