"""The few-row projection GEMM (csrc/kernels/gemm_skinny.hip) against fp32 PyTorch.  GPU only.

Shapes sit on the edges of its rules: one row and the most rows, shares of 4 columns that fill no row block,
one block, two and four (N / 256 above 16, 32), more than one workgroup per CU, K of one 128-byte line (fewer lines
than waves) up to the longest.  Bound: the output is one bf16 rounding (2^-9 of its value) of an fp32 sum over
K bf16 products, whose own error stays below 2^-9 of the sum's size at these K; with the norm, x * w is rounded
once more before the sum (2^-9 per term, averaging down).  2-norm over all outputs: 2^-8."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 8, 64), (3, 36, 128), (16, 896, 896), (7, 1152, 4864), (10, 4096, 8192), (16, 4100, 448), (4, 5120, 5120),
          (9, 8196, 576), (16, 18432, 4096), (2, 70000, 256), (5, 2048, 12288)]


@pytest.fixture(scope="module")
def ops():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops = get_ops("hip")
    if ops.gemm_plan.mode != "1":
        pytest.skip("BCG_HAND_GEMM")
    return ops


def _data(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N + K)
    x = (torch.randn(M, K, device="cuda", generator=g) * 3).to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).to(torch.bfloat16)
    nw = (1 + 0.2 * torch.randn(K, device="cuda", generator=g)).to(torch.bfloat16)
    return x, w, nw, g


def _off(out, ref):
    return ((out.double() - ref.double()).norm() / ref.double().norm()).item()


def _calls(ops, fn):
    log = ops.dispatch_log
    saved, log.enabled, log.calls = (log.enabled, log.calls), True, {}
    try:
        out = fn()
        return out, {k[5] for k in log.calls}
    finally:
        log.enabled, log.calls = saved


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_against_fp32(ops, M, N, K):
    x, w, nw, g = _data(M, N, K)
    bias = torch.randn(N, device="cuda", generator=g).to(torch.bfloat16)
    normed = (x.double() * torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + 1e-6)) * nw.double()
    y, yn = x.double() @ w.double().t(), normed @ w.double().t()
    out, used = _calls(ops, lambda: ops.linear(x, w, bias))
    assert used == {"skinnyx1"} and _off(out, y + bias.double()) < 2 ** -8
    assert torch.equal(out, ops.linear(x, w, bias))     # a fixed order of summation
    if K <= 8192:
        assert _off(ops.norm_linear(x, nw, 1e-6, w, bias), yn + bias.double()) < 2 ** -8
    res = torch.randn(M, N, device="cuda", generator=g).to(torch.bfloat16)
    want = y + res.double()
    assert ops.linear_residual(x, w, res) is res and _off(res, want) < 2 ** -8
    if N % 8 == 0:
        silu = torch.nn.functional.silu
        assert _off(ops.linear_silu(x, w), silu(y[:, :N // 2]) * y[:, N // 2:]) < 2 ** -7      # two factors
    if N % 8 == 0 and K <= 8192:
        assert _off(ops.norm_linear_silu(x, nw, 1e-6, w), silu(yn[:, :N // 2]) * yn[:, N // 2:]) < 2 ** -7


def test_other_forms_take_the_general_path(ops):
    """17 rows, a K off the 128-byte line or past the longest, strided and misaligned operands."""
    for M, N, K in [(17, 256, 256), (4, 256, 96)]:
        x, w, nw, _ = _data(M, N, K)
        out, used = _calls(ops, lambda: ops.norm_linear(x, nw, 1e-6, w))
        assert "skinnyx1" not in used
        ref = ops.linear(ops.rmsnorm(x, nw, 1e-6), w)
        assert torch.equal(out, ref)
    x, w, nw, _ = _data(4, 256, 12352)
    out, used = _calls(ops, lambda: ops.linear(x, w))
    assert "skinnyx1" not in used and _off(out, x.double() @ w.double().t()) < 2 ** -8
    with pytest.raises(RuntimeError):          # the norm's own limit: 8192 columns, for any number of rows
        ops.norm_linear(x[:, :8256].contiguous(), nw[:8256].contiguous(), 1e-6, w[:, :8256].contiguous())
    x, w, _, _ = _data(4, 64, 512)
    wide = torch.zeros(4, 1024, device="cuda", dtype=torch.bfloat16)
    wide[:, :512] = x
    flat = torch.zeros(64 * 512 + 4, device="cuda", dtype=torch.bfloat16)
    flat[4:] = w.flatten()
    for a, b in ((wide[:, :512], w), (x, flat[4:].view(64, 512))):
        out, used = _calls(ops, lambda: ops.linear(a, b))
        assert "skinnyx1" not in used and _off(out, x.double() @ w.double().t()) < 2 ** -8


def test_rows_with_infinities_and_nan(ops):
    """A row of its own: what one row holds never reaches another."""
    x, w, nw, _ = _data(8, 512, 512)
    clean = ops.norm_linear(x, nw, 1e-6, w)
    x[3, 7], x[5, 9] = float("inf"), float("nan")
    out = ops.norm_linear(x, nw, 1e-6, w)
    keep = [0, 1, 2, 4, 6, 7]
    assert torch.equal(out[keep], clean[keep]) and out[5].isnan().all() and out[3].isnan().any()
