"""Table-routed experts whose sum goes straight into the stream (csrc/kernels/seqmix_latent.hip, experts_post_norm_kernel; routes found by the position
kernel in small steps) against the separate launches, one fp32 rounding of the sums apart, and against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,E,top,W,ff", [(1, 8, 2, 64, 64), (3, 4, 1, 128, 64), (64, 8, 2, 2048, 512), (200, 5, 3, 320, 128), (1024, 4, 2, 192, 128),
                                          (1025, 4, 2, 192, 128), (130, 16, 8, 260, 64), (40, 12, 9, 64, 64)])
@pytest.mark.parametrize("post,pre", [("dyt", "copy"), ("rms", "dyt"), ("rms", None), ("dyt", "dyt")])
def test_against_separate_launches(T, E, top, W, ff, post, pre):
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops, g = get_ops("hip"), torch.Generator().manual_seed(T)
    rnd = lambda *s: torch.randn(*s, generator=g).to(DEV)
    norms = {"dyt": ("dyt", 0.6, rnd(W), rnd(W)), "rms": ("rms", rnd(W), 1e-5), "copy": ("copy",), None: None}
    up, down = (rnd(E, 2 * ff, W) * W ** -0.5).bfloat16(), (rnd(E, W, ff) * ff ** -0.5).bfloat16()
    h, x = rnd(T, W).bfloat16(), rnd(T, W)
    table = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(50)]).int()
    table[7] = -1   # (a token whose experts are not there)
    table = table.to(DEV)
    tokens = torch.randint(0, 50, (T,), generator=g).int()
    tokens[0] = 7
    if T > 2:
        tokens[2] = 60   # (past the table: no expert)
    tokens = tokens.to(DEV)
    x1, x2 = x.clone(), x.clone()
    want = ops.residual_post_norm(x1, ops.moe_experts(h, up, down, *ops.moe_table_route(tokens, table, top), "silu_gated"), norms[post], norms[pre], torch.bfloat16)
    got = ops.table_experts_post_norm(x2, h, up, down, tokens, table, top, "silu_gated", norms[post], norms[pre], torch.bfloat16)
    torch.testing.assert_close(x2, x1, rtol=2 ** -20, atol=2 ** -20)
    # in float64: y rounded to bf16 behind hidden values rounded up to three times, 2^-9 each
    u, d = up.double().view(E, ff // 16, 2, 16, W), down.double()
    gate, lin = u[:, :, 0].reshape(E, ff, W), u[:, :, 1].reshape(E, ff, W)   # (rows in alternating groups of 16)
    idx = ops.moe_table_route(tokens, table, top)[0].long()
    y = torch.zeros(T, W, dtype=torch.float64, device=DEV)
    for e in range(E):
        rows = (idx == e).any(1).nonzero()[:, 0]
        z = h[rows].double()
        y[rows] += (torch.nn.functional.silu(z @ gate[e].T) * (z @ lin[e].T)) @ d[e].T / top
    if post == "dyt":
        step = torch.tanh(0.6 * y) * norms[post][2].double() + norms[post][3].double()
    else:
        step = y / torch.sqrt((y * y).mean(1, keepdim=True) + 1e-5) * norms[post][1].double()
    assert (x2.double() - x.double() - step).norm() <= 2 ** -7 * step.norm()   # (both zero where no token has an expert)
    assert (got is None) == (pre is None)
    if pre is not None:
        torch.testing.assert_close(got.float(), want.float(), rtol=2 ** -7, atol=2 ** -7)


# more slots than the position kernel's threads hold (16 each), with few and with many experts
@pytest.mark.parametrize("T,E,top", [(8192, 8, 2), (8193, 8, 2), (17000, 3, 1), (9000, 200, 2)])
def test_every_slot_has_a_place(T, E, top):
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops, g = get_ops("hip"), torch.Generator().manual_seed(T)
    W, ff = 64, 128
    up, down = torch.zeros(E, ff, W), torch.zeros(E, W, ff)
    up[:, 0, 0], down[:, 0, 0] = 1, torch.arange(E)   # (an expert answers its number)
    h = torch.zeros(T, W)
    h[:, 0] = 1
    idx = torch.rand(T, E, generator=g).argsort(-1)[:, :top].int()
    idx[T // 2] = -1
    out = ops.moe_experts(h.bfloat16().to(DEV), up.bfloat16().to(DEV), down.bfloat16().to(DEV), idx.to(DEV), torch.ones(T, top).to(DEV), "relu2").cpu()
    assert torch.equal(out[:, 0], idx.clamp(min=0).sum(1).float())
