"""Expert products on position tiles of 256 rows (bcg_gemm_w4_grouped) against the same equations in float64.  GPU only.

Routings at the edges of the tiles: exactly the first size of the rule, a multiple of 256 rows per expert, remainders of 1 and
255, experts without a row, everything on two experts; widths that leave a partial last column tile.  Bound: hidden
values and rows are each one bf16 rounding (2^-9) of an fp32 sum; 2-norm of the error 2^-7."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _routing(kind, T, E, top, g):
    if kind == "even":
        return torch.rand(T, E, device="cuda", generator=g).argsort(-1)[:, :top].int().contiguous()
    if kind == "two":           # experts 1 and E - 1 take every row
        return torch.tensor([1, E - 1], dtype=torch.int32, device="cuda").expand(T, 2)[:, :top].contiguous()
    a = torch.zeros(T, dtype=torch.int32, device="cuda")    # expert 1: one row, expert 2: 255 rows, expert 0: the rest
    a[0], a[1:256] = 1, 2
    return torch.stack([a, torch.full_like(a, E - 1)], 1)[:, :top].contiguous()


def _exact(h, up, down, idx, w, kind, limit):
    h, up, down = h.double(), up.double(), down.double()
    out = torch.zeros_like(h)
    for j in range(idx.shape[1]):
        for e in range(up.shape[0]):
            t = (idx[:, j] == e).nonzero()[:, 0]
            z = h[t] @ up[e].T
            if kind == "relu2":
                z = z.clamp(min=0) ** 2
            else:
                z = z.view(len(t), up.shape[1] // 32, 2, 16)
                g, u = (z[:, :, i].reshape(len(t), up.shape[1] // 2) for i in range(2))
                if kind == "silu_gated":
                    z = torch.nn.functional.silu(g) * u
                else:
                    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
                    z = g * torch.sigmoid(1.702 * g) * (u + 1)
            out[t] += w[t, j].double()[:, None] * (z @ down[e].T)
    return out


@pytest.mark.parametrize("kind,limit", [("silu_gated", 0.0), ("clamped_glu", 1.5), ("relu2", 0.0)])
@pytest.mark.parametrize("routing,T,E,top,W,ff", [("even", 128, 4, 2, 64, 128), ("even", 1000, 5, 3, 320, 384), ("two", 512, 6, 2, 128, 256),
                                                  ("split", 700, 4, 2, 192, 128), ("even", 64, 1, 1, 256, 128)])
def test_wide_experts(kind, limit, routing, T, E, top, W, ff):
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    from byzantine_consensus_llm_agents_amd.ops.seqmix import WIDE_SLOTS
    assert T * top >= WIDE_SLOTS * E
    ops, g = get_ops("hip"), torch.Generator(device="cuda").manual_seed(T + W)
    bf = dict(device="cuda", generator=g)
    n_up = ff if kind == "relu2" else 2 * ff
    h = torch.randn(T, W, **bf).bfloat16()
    up, down = (torch.randn(E, n_up, W, **bf) * W ** -0.5).bfloat16(), (torch.randn(E, W, ff, **bf) * ff ** -0.5).bfloat16()
    idx, w = _routing(routing, T, E, top, g), torch.rand(T, top, **bf)
    want = _exact(h, up, down, idx, w, kind, limit)
    for _ in range(2):
        out = ops.moe_experts(h, up, down, idx, w, kind, limit)
        assert ((out.double() - want).norm() / want.norm()).item() < 2 ** -7


def test_a_row_reaches_no_other():
    """Padding rows of a tile hold whatever memory held: poison it."""
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops, g = get_ops("hip"), torch.Generator(device="cuda").manual_seed(3)
    T, E, W, ff = 300, 4, 128, 128
    h = torch.randn(T, W, device="cuda", generator=g).bfloat16()
    up, down = torch.randn(E, 2 * ff, W, device="cuda", generator=g).bfloat16(), torch.randn(E, W, ff, device="cuda", generator=g).bfloat16()
    idx, w = _routing("even", T, E, 2, g), torch.rand(T, 2, device="cuda", generator=g)
    clean = ops.moe_experts(h, up, down, idx, w, "silu_gated")
    cap = (T * 2 + E * 255 + 255) // 256 * 256
    poison = [torch.full((cap, n), float("nan"), device="cuda", dtype=torch.bfloat16) for n in (W, ff)]
    del poison
    assert torch.equal(ops.moe_experts(h, up, down, idx, w, "silu_gated"), clean)
