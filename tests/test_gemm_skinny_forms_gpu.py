"""The few-row projection GEMM (csrc/kernels/gemm_skinny.hip) past its first form: two blocks of rows, several passes of a
workgroup, half a unit of K at the end of a row, long rows, fp8 operands.  Against float64.  GPU only.

Bounds as in test_gemm_skinny_gpu.py: one bf16 rounding (2^-9) of an fp32 sum whose own error stays below 2^-9: 2^-8 in the
2-norm; the gated unit has two factors.  fp8 operands are exact in float64, so the same holds."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows, N, K: 17, 32, 33, 48, 49 and 64 rows; one column group per workgroup; passes (N / 256 > 64 at two blocks, > 128 at one); K of 1, 1.5 and
# an odd number of units; K from 12289 on and the longest
SHAPES = [(17, 8, 128), (32, 1028, 192), (20, 5120, 5120), (31, 17408, 448), (24, 70000, 320), (32, 4096, 17408), (16, 70000, 1088),
          (10, 5120, 17408), (3, 256, 32768), (16, 520, 1600), (32, 36864, 576), (33, 8, 64), (48, 8192, 320), (49, 1024, 2048), (64, 8188, 1088)]


@pytest.fixture(scope="module")
def ops():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops = get_ops("hip")
    if ops.gemm_plan.mode != "1":
        pytest.skip("BCG_HAND_GEMM")
    return ops


def _off(out, ref):
    return ((out.double() - ref).norm() / ref.norm()).item()


def _calls(ops, fn):
    log = ops.dispatch_log
    saved, log.enabled, log.calls = (log.enabled, log.calls), True, {}
    try:
        out = fn()
        return out, {k[5] for k in log.calls}
    finally:
        log.enabled, log.calls = saved


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_bf16(ops, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N + K)
    x = (torch.randn(M, K, device="cuda", generator=g) * 3).to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).to(torch.bfloat16)
    bias = torch.randn(N, device="cuda", generator=g).to(torch.bfloat16)
    y = x.double() @ w.double().t()
    out, used = _calls(ops, lambda: ops.linear(x, w, bias))
    assert all(u.startswith("skinny") for u in used) and len(used) == 1
    assert _off(out, y + bias.double()) < 2 ** -8 and torch.equal(out, ops.linear(x, w, bias))
    res = torch.randn(M, N, device="cuda", generator=g).to(torch.bfloat16)
    want = y + res.double()
    assert ops.linear_residual(x, w, res) is res and _off(res, want) < 2 ** -8
    if N % 8 == 0:
        gated = torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
        assert _off(ops.linear_silu(x, w), gated) < 2 ** -7


# rows of 8, 16 and 32 KB: other orders of K
@pytest.mark.parametrize("M,N,K", [(1, 256, 4096), (4, 2048, 4096), (16, 1028, 4096), (1, 520, 8192), (5, 8192, 8192), (20, 4096, 8192), (3, 1024, 16384),
                                   (16, 4096, 16384), (24, 5120, 16384)])
def test_row_pitches(ops, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    x = (torch.randn(M, K, device="cuda", generator=g) * 3).to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).to(torch.bfloat16)
    y = x.double() @ w.double().t()
    out, used = _calls(ops, lambda: ops.linear(x, w))
    assert all(u.startswith("skinny") for u in used) and _off(out, y) < 2 ** -8 and torch.equal(out, ops.linear(x, w))
    if M <= 16 and K <= 8192:
        nw = (1 + 0.3 * torch.randn(K, device="cuda", generator=g)).to(torch.bfloat16)
        xd = x.double()
        normed = xd * torch.rsqrt(xd.square().mean(1, keepdim=True) + 1e-6) * nw.double()
        assert _off(ops.norm_linear(x, nw, 1e-6, w), normed @ w.double().t()) < 2 ** -7   # (the norm rounds its products too)
    if N % 16 == 0 and (K <= 4096 or N >= 4096):     # (of bytes that are twice as many)
        f8 = torch.float8_e4m3fn
        xq, wq = (x * 20).to(f8), (w * 100).to(f8)
        xq, wq = torch.cat([xq, xq], 1), torch.cat([wq, wq], 1)
        xs, ws = torch.full((M, 1), 0.05, device="cuda"), torch.full((N,), 0.01, device="cuda")
        ref = (xq.double() @ wq.double().t()) * 0.05 * 0.01
        assert _off(ops.linear_fp8(xq, xs, wq, ws), ref) < 2 ** -8


@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (16, 1024, 640), (17, 528, 384), (20, 8192, 6144), (32, 36864, 896), (9, 70000, 256),
                                   (32, 6144, 16384)])
def test_fp8(ops, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N + K)
    f8 = torch.float8_e4m3fn
    xq = torch.randn(M, K, device="cuda", generator=g).mul_(100).clamp_(-448, 448).to(f8)
    wq = torch.randn(N, K, device="cuda", generator=g).mul_(100).clamp_(-448, 448).to(f8)
    xs = torch.rand(M, 1, device="cuda", generator=g) * 0.01 + 0.001
    ws = (torch.rand(N, device="cuda", generator=g) + 0.1) * K ** -0.5
    y = (xq.double() @ wq.double().t()) * xs.double() * ws.double()
    bias = torch.randn(N, device="cuda", generator=g).to(torch.bfloat16)
    out, used = _calls(ops, lambda: ops.linear_fp8(xq, xs, wq, ws, bias))
    assert all(u.startswith("skinny") for u in used) and len(used) == 1
    assert _off(out, y + bias.double()) < 2 ** -8 and torch.equal(out, ops.linear_fp8(xq, xs, wq, ws, bias))
    res = torch.randn(M, N, device="cuda", generator=g).to(torch.bfloat16)
    want = y + res.double()
    assert ops.linear_fp8_residual(xq, xs, wq, ws, res) is res and _off(res, want) < 2 ** -8


def test_nothing_is_read_past_the_operands(ops):
    """Rows past M and N, and the second half of a last unit, are what lies behind: infinities there leave no trace."""
    for M, N, K in ((3, 36, 320), (18, 100, 192), (10, 1000, 2112)):
        g = torch.Generator(device="cuda").manual_seed(N)
        xb = torch.full(((M + 32) * K,), float("inf"), device="cuda", dtype=torch.bfloat16)
        wb = torch.full(((N + 128) * K,), float("inf"), device="cuda", dtype=torch.bfloat16)
        x, w = xb[:M * K].view(M, K), wb[:N * K].view(N, K)
        x.copy_(torch.randn(M, K, device="cuda", generator=g))
        w.copy_(torch.randn(N, K, device="cuda", generator=g))
        assert _off(ops.linear(x, w), x.double() @ w.double().t()) < 2 ** -8


def test_norm_weight_infinities(ops):
    """An infinite norm weight reaches what it is multiplied with and nothing else (K that ends inside a turn of the waves)."""
    x = torch.ones(2, 1088, device="cuda", dtype=torch.bfloat16)
    w = torch.ones(64, 1088, device="cuda", dtype=torch.bfloat16)
    nw = torch.ones(1088, device="cuda", dtype=torch.bfloat16)
    nw[-1] = float("inf")
    assert (ops.norm_linear(x, nw, 1e-6, w) == float("inf")).all()


@pytest.mark.parametrize("M,K,N,KW", [(4, 256, 64, 512), (20, 512, 128, 1024), (32, 128, 4096, 256)])
def test_fp8_operands_of_other_rows_are_refused(ops, M, K, N, KW):
    """Rows of W that are longer than those of x: an error before any launch, on both entry points."""
    f8 = torch.float8_e4m3fn
    xq, wq = torch.zeros(M, K, device="cuda").to(f8), torch.zeros(N, KW, device="cuda").to(f8)
    xs, ws = torch.ones(M, 1, device="cuda"), torch.ones(N, device="cuda")
    res = torch.ones(M, N, device="cuda", dtype=torch.bfloat16)
    with pytest.raises(ValueError):
        ops.linear_fp8_residual(xq, xs, wq, ws, res)
    with pytest.raises(ValueError):
        ops.linear_fp8(xq, xs, wq, ws)
    assert (res == 1).all()
