"""The recurrences' workgroups over heads and segments ordered by length (csrc/kernels/seqmix_common.h, segment_of): every segment is taken once, whatever
the order of the lengths is, up to and past the 64 segments that are ordered.  Against 64-bit arithmetic, bounds of the kernels' own tests."""
import pytest
import torch

import padadra_cases as C
from test_delta_scan_gpu import _exact

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# equal lengths among them; 64, 65 and 70 segments
@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("B,H,e", [(1, 9, 40), (3, 16, 70), (8, 8, 130), (64, 2, 33), (65, 9, 16), (70, 3, 65)])
def test_every_segment_once(delta, B, H, e):
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops = get_ops("hip")
    gen = torch.Generator().manual_seed(B)
    # (chunks are taken from 16 tokens on where a step does not say its longest segment)
    parts = [(int(torch.randint(0, 2, (1,), generator=gen)) * 5, n) for n in torch.randint(16, 24, (B,), generator=gen).tolist()]
    parts[B // 2] = (0, 70)
    rows = torch.randperm(B + 1, generator=gen)[:B].tolist()
    mc, md = C.segments(parts, rows), C.segments(parts, rows, DEV)
    T, d = mc.positions.numel(), 32
    q, k = (torch.nn.functional.normalize(torch.randn(T, H, d, generator=gen), dim=-1) for _ in range(2))
    g = torch.exp(-torch.rand(T, H, 1, generator=gen))
    v = torch.randn(T, H * e, generator=gen)
    beta = torch.rand(T, H, generator=gen)
    state = torch.randn(B + 1, H, d, e, generator=gen)
    if delta:
        want, moved = _exact(q, k, g, v, beta, mc, state)
    else:
        from byzantine_consensus_llm_agents_amd.ops import reference as ref
        moved = state.double()
        want = ref.gated_state_scan(q.double(), k.double(), g.double(), v.double(), beta.double(), mc, moved, False)
    sd = state.to(DEV)
    got = ops.gated_state_scan(q.to(DEV), k.to(DEV), g.to(DEV), v.to(DEV), beta.to(DEV), md, sd, delta)
    bound = dict(atol=2.0 ** -24 * (d + 8) * 70 / 2, rtol=2.0 ** -20)
    torch.testing.assert_close(got.cpu().double(), want.double(), **bound)
    torch.testing.assert_close(sd.cpu().double(), moved.double(), **bound)
