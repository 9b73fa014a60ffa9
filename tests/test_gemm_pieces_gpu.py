"""Prefill-sized projections at row counts the table does not hold (`GemmPlan.pieces`): rows split between two
kernels, or the 256 x 256 kernel in the library's place.  GPU only.  Bound: one bf16 rounding (2^-9) of an fp32
sum; 2-norm of the error 2^-8 (2^-7 with the gated unit, a product of two)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

W4 = (11, 1)
# M, N, K, epi, runs of rows (None: the library)
CASES = [(4449, 4096, 12288, 2, [4096, 353]),      # one whole round of tiles, then 353 rows
         (4097, 4096, 8192, 2, [4096, 1]),         # ... then one row
         (4449, 4096, 12288, 0, [4096, 353]), (2049, 8192, 4096, 0, [2048, 1]),
         (2560, 32768, 1024, 0, [2560]),           # whole rounds: one run, the library
         (8183, 11264, 2048, 0, [8183]), (2900, 24576, 512, 0, [2900]),
         (2048, 1792, 1024, 1, [2048]), (2177, 9728, 896, 1, [2177]),
         (2565, 12800, 896, 0, [2560, 5]), (8706, 7680, 896, 2, [8704, 2])]   # rounds full but for a few tiles on the library


@pytest.mark.parametrize("M,N,K,epi,rows", CASES)
def test_pieces(M, N, K, epi, rows):
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops = get_ops("hip")
    if ops.gemm_plan.mode != "1":
        pytest.skip("BCG_HAND_GEMM")
    assert [r for r, _ in ops.gemm_plan.pieces(M, N, K, epi)] == rows
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    y = (x.float() @ w.float().t()).double()
    off = lambda a, b: ((a.double() - b).norm() / b.norm()).item()  # noqa: E731
    if epi == 0:
        bias = torch.randn(N, device="cuda", generator=g).bfloat16()
        assert off(ops.linear(x, w), y) < 2 ** -8 and off(ops.linear(x, w, bias), y + bias.double()) < 2 ** -8
    elif epi == 1:
        assert off(ops.linear_silu(x, w), torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]) < 2 ** -7
    else:
        res = torch.randn(M, N, device="cuda", generator=g).bfloat16()
        want = y + res.double()
        assert ops.linear_residual(x, w, res) is res and off(res, want) < 2 ** -8


def test_operands_that_do_not_lie_so():
    """A transposed weight, an offset of 8 bytes, a strided residual and an operand with a gradient keep the library."""
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops, M, N, K = get_ops("hip"), 8183, 11264, 256
    assert ops.gemm_plan.pieces(M, N, K, 0)[0][1] == W4 or ops.gemm_plan.mode != "1"
    x, w = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(N, K, device="cuda").bfloat16() * K ** -0.5
    want = x.float() @ w.float().t()
    off = lambda a, b: ((a.float() - b).norm() / b.norm()).item()  # noqa: E731
    flat = torch.zeros(M * K + 4, device="cuda", dtype=torch.bfloat16)
    flat[4:] = x.flatten()
    assert off(ops.linear(x, w.t().contiguous().t()), want) < 2 ** -8
    assert off(ops.linear(flat[4:].view(M, K), w), want) < 2 ** -8
    res = torch.zeros(M, 2 * N, device="cuda", dtype=torch.bfloat16)
    assert off(ops.linear_residual(x, w, res[:, :N]), want) < 2 ** -8 and not res[:, N:].any()
    xg = x.clone().requires_grad_()
    ops.linear(xg, w).float().sum().backward()
    assert off(xg.grad, w.float().sum(0).expand(M, K)) < 2 ** -7


# M, N, K, columns of the whole rounds (N: one launch)
COLUMNS = [(448, 34816, 512, 32768), (333, 34816, 64, 32768), (300, 34816, 64, 34816), (512, 33792, 128, 32768), (600, 22528, 256, 21760),
           (768, 22016, 192, 21760), (448, 32768, 128, 32768), (256, 66048, 64, 66048), (600, 24576, 128, 24576), (448, 34832, 64, 34832)]


@pytest.mark.parametrize("M,N,K,n1", COLUMNS)
def test_columns(M, N, K, n1):
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops = get_ops("hip")
    if ops.gemm_plan.mode != "1":
        pytest.skip("BCG_HAND_GEMM")
    assert ops.gemm_plan.columns(M, N, K) == n1
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    y = (x.float() @ w.float().t()).double()
    want = torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
    got = ops.linear_silu(x, w)
    assert ((got.double() - want).norm() / want.norm()).item() < 2 ** -7
    # the last features alone (the rest's tiles)
    assert ((got[:, -64:].double() - want[:, -64:]).norm() / want[:, -64:].norm()).item() < 2 ** -7
