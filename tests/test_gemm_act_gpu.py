"""Projections with a feed-forward's activation in the epilogue of the 256 x 256 kernel (csrc/kernels/gemm_w4.hip, epilogues 5
and 6) against 64-bit products, at the edges of its tiles, and the rule that takes a call there against the two-pass form."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    o = get_ops("hip")
    o.prepare_device(torch.device(DEV))
    return o


def _operands(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g) * 3 / K ** 0.5).to(torch.bfloat16)   # products of about 3: the clamp at 4 is met
    z = x.double() @ w.double().t()
    dz = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())   # fp32 sums of K products
    return x.to(DEV), w.to(DEV), z, dz


def _close(got, want, slack):
    """One rounding to bf16 (2^-9, twice that) and `slack`."""
    bound = 2.0 ** -8 * want.abs() + slack + 2.0 ** -20
    assert ((got.double().cpu() - want).abs() <= bound).all()


# one row, one short of a tile, one past it, three row tiles; one column tile of either side, several, K of one and many tiles
@pytest.mark.parametrize("M,inter,K", [(1, 128, 64), (255, 128, 128), (257, 384, 192), (600, 640, 1024)])
def test_clamped(ops, monkeypatch, M, inter, K):
    monkeypatch.setattr(ops.gemm_plan, "clamped_tiles", lambda *a: True)
    x, w, z, dz = _operands(M, 2 * inter, K, M)
    limit = 4.0
    g, u = z[:, :inter].clamp(max=limit), z[:, inter:].clamp(-limit, limit)
    want = g * torch.sigmoid(1.702 * g) * (u + 1)
    # slope of g sigmoid(1.702 g): at most 1.1, of u + 1: limit; the unit of the smallest g keeps 2^-20 of them
    slack = 1.1 * (limit + 1) * dz[:, :inter] + limit * dz[:, inter:] + 2.0 ** -20 * (limit + 1) * g.abs()
    _close(ops.linear_clamped_glu(x, w, limit), want, slack)


@pytest.mark.parametrize("M,at,N,K", [(1, 256, 272, 64), (255, 256, 512, 128), (257, 512, 1296, 192), (600, 768, 2048, 1024)])
def test_tail(ops, monkeypatch, M, at, N, K):
    monkeypatch.setattr(ops.gemm_plan, "tail_tiles", lambda *a: True)
    x, w, z, dz = _operands(M, N, K, M)
    y, hidden = ops.linear_tail_gelu(x, w, at)
    _close(y, z[:, :at], dz[:, :at])
    tail = z[:, at:]
    _close(hidden, torch.nn.functional.gelu(tail, approximate="tanh"), 1.13 * dz[:, at:] + 2.0 ** -20 * tail.abs())


def test_clamped_wide_output(ops):
    """Twice the output's columns are past 32-bit offsets, the output is not: 16384 x 32768 of 64."""
    M, inter, K, limit = 16384, 32768, 64, 4.0
    assert ops.gemm_plan.clamped_tiles(M, 2 * inter, K)
    x = torch.randn(M, K, device=DEV, generator=torch.Generator(DEV).manual_seed(1)).to(torch.bfloat16)
    w = (torch.randn(2 * inter, K, device=DEV, generator=torch.Generator(DEV).manual_seed(2)) * 3 / K ** 0.5).to(torch.bfloat16)
    out = ops.linear_clamped_glu(x, w, limit)
    rows = torch.tensor([0, 255, 256, 8191, 16383], device=DEV)
    z = x[rows].double() @ w.double().t()
    dz = K * 2.0 ** -24 * (x[rows].double().abs() @ w.double().abs().t())
    g, u = z[:, :inter].clamp(max=limit), z[:, inter:].clamp(-limit, limit)
    slack = 1.1 * (limit + 1) * dz[:, :inter] + limit * dz[:, inter:] + 2.0 ** -20 * (limit + 1) * g.abs()
    _close(out[rows], (g * torch.sigmoid(1.702 * g) * (u + 1)).cpu(), slack.cpu())


def test_extremes(ops, monkeypatch):
    """Infinities and values whose exponentials overflow come out as in the passes of their own."""
    for name in ("clamped_tiles", "tail_tiles"):
        monkeypatch.setattr(ops.gemm_plan, name, lambda *a: True)
    x = torch.zeros(8, 64, dtype=torch.bfloat16, device=DEV)
    x[:, 0] = torch.tensor([0.0, 300.0, -300.0, 1e30, -1e30, float("inf"), float("-inf"), float("nan")])
    w = torch.zeros(512, 64, dtype=torch.bfloat16, device=DEV)
    w[:, 0] = 1.0
    both = ops.linear(x, w)
    torch.testing.assert_close(ops.linear_clamped_glu(x, w, 7.0), ops.gated_act(both, "clamped_glu", 7.0), rtol=2 ** -7, atol=0, equal_nan=True)
    torch.testing.assert_close(ops.linear_tail_gelu(x, w, 256)[1], ops.act_fn(both[:, 256:], "gelu_tanh"), rtol=2 ** -7, atol=0, equal_nan=True)


def test_routes(ops):
    """Both sides of the rules and operands that only the library takes: the two-pass form's values."""
    K, ff, at = 1024, 4096, 1024
    x, w, _, _ = _operands(1030, at + ff, K, 1)
    assert not ops.gemm_plan.clamped_tiles(300, 2 * ff, K) and ops.gemm_plan.clamped_tiles(2048, 2 * ff, K)
    assert not ops.gemm_plan.tail_tiles(1030, at + ff, K, at) and ops.gemm_plan.tail_tiles(3000, at + ff, K, at)
    x2 = torch.cat([x, x, x])[:3000]
    up = torch.cat([w, w])[:2 * ff]
    wide = torch.cat([x2, x2], 1)[:, :K]   # rows of another stride
    for a in (x2, wide):
        want = ops.gated_act(ops.linear(a, up), "clamped_glu", 4.0).float()
        # two roundings of either factor before the product against none: 2^-8 each, and the clamp's corner
        torch.testing.assert_close(ops.linear_clamped_glu(a, up, 4.0).float(), want, rtol=2 ** -6, atol=2 ** -5)
        y, hidden = ops.linear_tail_gelu(a, w, at)
        both = ops.linear(a, w)
        assert (hidden is None) == (a is wide)
        torch.testing.assert_close(y[:, :at].float(), both[:, :at].float(), rtol=2 ** -7, atol=2 ** -7)
        if hidden is not None:
            torch.testing.assert_close(hidden.float(), ops.act_fn(both[:, at:], "gelu_tanh").float(), rtol=2 ** -6, atol=2 ** -6)
    with pytest.raises(ValueError):
        ops.linear_clamped_glu(x2, up, 0.0)
