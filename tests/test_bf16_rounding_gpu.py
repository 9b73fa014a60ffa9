"""The kernels' rounding from fp32 to bf16 against torch's, bit by bit.  GPU only."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_every_kind_of_value():
    """Ties, neighbours of ties, zeros, the largest numbers, infinities and NaN, through a copy of the stream in bf16.  The kernels are built
    with subnormal numbers flushed: those are zeros."""
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops, W = get_ops("hip"), 4096
    high = torch.arange(1 << 16, dtype=torch.int64)                          # every bf16 value, and around the middle to the next
    bits = torch.stack([high * 65536 + low for low in (0, 1, 0x7fff, 0x8000, 0x8001, 0xffff)])
    bits = torch.cat([bits.flatten(), torch.randint(0, 1 << 32, (1 << 18,), generator=torch.Generator().manual_seed(0))])
    x = (bits - ((bits >> 31) << 32)).to(torch.int32).cuda().view(torch.float32).view(-1, W)
    zeros, w = torch.zeros(x.shape, device="cuda", dtype=torch.bfloat16), torch.ones(W, device="cuda")
    want = torch.where(x.abs() < 2.0 ** -126, torch.zeros_like(x), x).bfloat16()
    got = ops.residual_post_norm(x.clone(), zeros, ("rms", w, 1e-5), ("copy",), torch.bfloat16)
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)
    assert torch.equal(got.view(torch.int16)[~nan], want.view(torch.int16)[~nan])
