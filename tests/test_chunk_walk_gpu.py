"""The walk over chunks (csrc/kernels/seqmix_retention.hip) at its remainders, in workgroups of 16, 32 and 64 value columns: lengths around blocks of 16 and
chunks of 64 tokens, decays of 0 and 1 among them, and an infinite last key.  Against 64-bit arithmetic."""
import math

import pytest
import torch

import padadra_cases as C

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(n, H, d, e, per_token, seed):
    gen = torch.Generator().manual_seed(seed)
    q, k = (torch.nn.functional.normalize(torch.randn(n, 1, d, generator=gen), dim=-1) for _ in range(2))
    g = torch.exp(-torch.rand(n, H, 1, generator=gen)) if per_token else torch.linspace(0.0, 1.0, H)
    if per_token:
        g[n // 2] = 0.0
    return q, k, g, torch.randn(n, H * e, generator=gen), torch.randn(2, H, d, e, generator=gen)


def _run(q, k, g, v, state, n):
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    sd = state.to(DEV)
    got = get_ops("hip").gated_state_scan(q.to(DEV), k.to(DEV), g.to(DEV), v.to(DEV), None, C.segments([(5, n)], [1], DEV), sd, False)
    return got.cpu(), sd.cpu()


@pytest.mark.parametrize("H,e", [(2, 48), (129, 48), (257, 64)])   # 16, 32 and 64 columns per workgroup
@pytest.mark.parametrize("per_token", [True, False])
@pytest.mark.parametrize("n", [63, 64, 65, 79, 80, 81, 145])
def test_remainders(H, e, per_token, n):
    from byzantine_consensus_llm_agents_amd.ops import reference as ref
    d = 32
    q, k, g, v, state = _inputs(n, H, d, e, per_token, n)
    moved = state.double()
    want = ref.gated_state_scan(q.double(), k.double(), g.double(), v.double(), None, C.segments([(5, n)], [1]), moved, False)
    got, sd = _run(q, k, g, v, state, n)
    # (sums of at most n terms of about 1 and a state of d of them, in fp32 chains of 16)
    bound = dict(atol=2.0 ** -24 * (d + 8) * math.sqrt(n), rtol=2.0 ** -20)
    torch.testing.assert_close(got.double(), want.double(), **bound)
    torch.testing.assert_close(sd.double(), moved, **bound)


@pytest.mark.parametrize("H,e", [(2, 48), (129, 48), (257, 64)])
@pytest.mark.parametrize("n", [70, 130])
def test_an_infinite_last_key_stays_in_its_feature(H, e, n):
    d = 32
    q, k, g, v, state = _inputs(n, H, d, e, True, n)
    clean, kept = _run(q, k, g, v, state, n)
    k[-1, 0, 3] = math.inf
    got, sd = _run(q, k, g, v, state, n)
    assert torch.equal(got[:-1], clean[:-1])
    others = [f for f in range(d) if f != 3]
    assert torch.equal(sd[1][:, others], kept[1][:, others])
    assert torch.equal(sd[1][:, 3], torch.sign(v[-1].view(H, e)) * math.inf)
