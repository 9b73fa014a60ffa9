"""Row-wise fp8 quantisation has the bits of a division by the row's scale, at the quotients that are ties between two e4m3 values too."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    return get_ops("hip")


def _divided(x):
    """(bytes, scales) of bf16 rows, by IEEE division and torch's rounding, on the CPU."""
    x = x.float().cpu()
    s = x.abs().amax(-1).clamp(min=1e-12) / 448.0
    return (x / s[:, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8), s


def _all_mantissas(top):
    """Row m: maximum (1 + m / 128) 2^top, and every bf16 value of both signs below it over 15 powers of two, and zeros of both signs."""
    m = 1.0 + torch.arange(128) / 128.0
    values = torch.cat([m * 2.0 ** (top - k) for k in range(15)])
    values = torch.cat([values, -values])
    rows = torch.where(values.abs()[None] <= (m * 2.0 ** top)[:, None], values[None], values[None] * 0.0)
    return rows.to(torch.bfloat16)


def _same(q, s, x):
    want, s_want = _divided(x)
    torch.testing.assert_close(s.cpu(), s_want, atol=0, rtol=0)
    off = (q.view(torch.uint8).cpu() != want).nonzero()
    assert not len(off), (len(off), off[0].tolist())


@pytest.mark.parametrize("top", [-30, 0, 5, 100])
def test_quant_all_mantissas(hip, top):
    x = _all_mantissas(top)
    _same(*hip.quant_fp8(x.cuda()), x)


@pytest.mark.parametrize("I", [3840, 65536])   # (in registers, read twice)
def test_silu_mul_all_mantissas(hip, I):
    x = _all_mantissas(3).repeat(1, -(-I // 3840))[:, :I]
    gate = torch.full_like(x, 64.0)   # silu(64) is 64 in 24 bits
    _same(*hip.silu_mul_fp8(torch.cat([gate, x / 64.0], 1).contiguous().cuda()), x)


@pytest.mark.parametrize("T", [200, 300])
def test_norm_rows(hip, T):
    torch.manual_seed(3)
    x = torch.randn(T, 6144, dtype=torch.bfloat16, device="cuda")
    w = (torch.rand(6144, device="cuda") + 0.5).to(torch.bfloat16)
    q, s = hip.rmsnorm_fp8(x, w, 1e-5)
    y = hip.rmsnorm(x, w, 1e-5)   # (a sum in another order may round a value the other way: rows where it did differ in it and perhaps the scale)
    want, s_want = _divided(y)
    differ = (q.view(torch.uint8).cpu() != want).float().mean(1)
    assert (differ < 2.0 / 6144).float().mean() > 0.9


def test_infinite_maximum(hip):
    x = torch.randn(3, 512, dtype=torch.bfloat16)
    x[1, 77] = float("inf")
    q, s = hip.quant_fp8(x.cuda())
    assert s.cpu()[1] == float("inf")
    finite = torch.arange(512) != 77
    assert not (q.view(torch.uint8).cpu()[1, finite] & 0x7f).any()   # a finite value over infinity is zero
    keep = torch.tensor([0, 2])
    assert torch.equal(q.view(torch.uint8).cpu()[keep], _divided(x[keep])[0])


def test_silu_is_divided(hip):
    """silu(-88) u with u = 2^100: 1 + exp(88) has a reciprocal below the smallest normal number, the quotient has not."""
    gu = torch.cat([torch.full((2, 64), -88.0), torch.full((2, 64), 2.0 ** 100)], 1).to(torch.bfloat16)
    q, s = hip.silu_mul_fp8(gu.cuda())
    want = -88.0 / (1.0 + torch.exp(torch.tensor(88.0, dtype=torch.float64))) * 2.0 ** 100
    got = q.float().cpu().double() * s.cpu().double()[:, None]
    assert ((got / want - 1.0).abs() < 2.0 ** -8).all()   # (the row's maximum: one rounding to bf16, 448 in e4m3)
