"""The delta-rule recurrence with one decay per head (csrc/kernels/seqmix_state.hip, delta_scan_kernel) against 64-bit arithmetic:
chunks of tokens with remainders, row and column edges, single tokens among longer segments, decays of 1, tiny and 0."""

import pytest
import torch

import padadra_cases as C

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _exact(q, k, g, v, beta, meta, state):
    T, H = beta.shape
    per, e = H // q.shape[1], state.shape[3]
    q, k = (x.double().repeat_interleave(per, 1) for x in (q, k))
    v, out, state = v.double().view(T, H, e), torch.zeros(T, H, e, dtype=torch.float64), state.double()
    for b, row in enumerate(meta.state_rows.tolist()):
        s, n = meta.q_start[b:b + 2].tolist()
        S = state[row] * float(meta.positions[s] != 0)
        for t in range(s, n):
            S = S * g[t].double()[:, :, None]
            u = beta[t].double()[:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
            S = S + k[t][:, :, None] * u[:, None, :]
            out[t] = (S * q[t][:, :, None]).sum(1)
        state[row] = S
    return out, state


# (position, tokens) per segment: whole chunks of 8 (4 past 128 rows), one more, one fewer, single tokens
PARTS, ROWS = [(0, 16), (7, 9), (3, 1), (0, 31), (40, 8), (0, 1)], [3, 0, 4, 1, 2, 6]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,Gq,d,e", [(4, 4, 32, 32), (2, 1, 20, 33), (6, 3, 64, 31), (4, 2, 48, 72), (4, 2, 128, 128), (3, 3, 100, 130), (2, 1, 256, 40),
                                      (1, 1, 1, 1), (64, 1, 130, 65)])   # (the last: more workgroups than the rule takes past 128 rows, in fp32)
def test_against_64_bits(dtype, H, Gq, d, e):
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops = get_ops("hip")
    gen = torch.Generator().manual_seed(d + e)
    mc, md = C.segments(PARTS, ROWS), C.segments(PARTS, ROWS, DEV)
    T = mc.positions.numel()
    assert T >= 4 * len(PARTS)
    q, k = (torch.nn.functional.normalize(torch.randn(T, Gq, d, generator=gen), dim=-1) for _ in range(2))
    g = torch.exp(-torch.rand(T, H, 1, generator=gen))
    g[::5], g[::7], g[::11] = 1.0, 1e-30, 0.0
    v = torch.randn(T, H * e + 5, generator=gen).to(dtype)[:, 2:2 + H * e]
    beta = torch.rand(T, H, generator=gen)
    state = torch.randn(8, H, d, e, generator=gen)
    want, moved = _exact(q, k, g, v, beta, mc, state)
    sd = state.to(DEV)
    got = ops.gated_state_scan(q.to(DEV), k.to(DEV), g.to(DEV), v.to(DEV), beta.to(DEV), md, sd, True)
    # unit k and q: a token's sums have d products and 8 roundings more, of partial sums about 1 (half an ulp 2^-24); at most 31
    # tokens pass them on, the decays forget half
    bound = dict(atol=2.0 ** -24 * (d + 8) * 31 / 2, rtol=2.0 ** -20)
    torch.testing.assert_close(got.cpu().double(), want, **bound)
    torch.testing.assert_close(sd.cpu().double(), moved, **bound)   # rows 5 and 7 untouched


def test_values_that_are_not_finite_stay_in_their_column():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops = get_ops("hip")
    md = C.segments([(0, 11)], [0], DEV)
    gen = torch.Generator(device=DEV).manual_seed(0)
    q, k = (torch.randn(11, 1, 24, generator=gen, device=DEV) for _ in range(2))
    g, beta = torch.full((11, 1, 1), 0.9, device=DEV), torch.full((11, 1), 0.5, device=DEV)
    v = torch.randn(11, 40, generator=gen, device=DEV)
    state = torch.zeros(1, 1, 24, 40, device=DEV)
    clean = ops.gated_state_scan(q, k, g, v, beta, md, state.clone(), True)
    v[3, 7], v[5, 9] = float("nan"), float("inf")
    got = ops.gated_state_scan(q, k, g, v, beta, md, state, True)
    other = torch.ones(40, dtype=torch.bool, device=DEV)
    other[[7, 9]] = False
    assert torch.equal(got[..., other], clean[..., other]) and torch.equal(got[:3], clean[:3])
    assert not got[3:, 0, 7].isfinite().any() and not got[5:, 0, 9].isfinite().any()
