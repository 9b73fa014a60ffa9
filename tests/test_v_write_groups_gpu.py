"""V^T of a packed step in the paged cache (csrc/kernels/rope_kv.hip, v_write_group_kernel): every token's column, and nothing else,
wherever the prompts' pages lie against the workgroups' 16 tokens."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (tokens, slot of the first inside its page) per sequence
STEPS = {
    "aligned": [(64, 0), (32, 0)],
    "shifted": [(21, 0), (50, 0), (17, 0), (33, 0)],                 # groups begin anywhere in a workgroup's tokens
    "resumed": [(15, 7), (47, 1), (16, 15), (40, 9)],                # the first page is partly filled already
    "single tokens": [(1, i % 16) for i in range(37)] + [(40, 0)],   # many groups in a workgroup's tokens
    "one short of a group": [(79, 0)], "one past it": [(65, 0)],
}


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("page", [8, 16, 32])
@pytest.mark.parametrize("step", STEPS)
def test_every_token_once(hd, page, step):
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops = get_ops("hip")
    g = torch.Generator().manual_seed(1)
    n_q, n_kv, L, layer = 3, 2, 2, 1
    first, slots, positions = 0, [], []
    need = [-(-(n + at) // page) for n, at in STEPS[step]]
    pages = torch.randperm(sum(need) + 2, generator=g)
    for (n, at), k in zip(STEPS[step], need):
        p = at + torch.arange(n)
        slots.append(pages[first:first + k][p // page] * page + p % page)
        positions.append(p)
        first += k
    slots, positions = torch.cat(slots), torch.cat(positions)
    T, NB = slots.numel(), pages.numel()
    qkv = torch.randn(T, (n_q + 2 * n_kv) * hd, generator=g).to(torch.bfloat16)
    k_cache = torch.zeros(L, NB, n_kv, page, hd, dtype=torch.bfloat16, device=DEV)
    v_cache = torch.full((L, NB, n_kv, hd, page), 7.0, dtype=torch.bfloat16, device=DEV)
    want = v_cache.cpu().clone()
    want[layer, slots // page, :, :, slots % page] = qkv.view(T, -1, hd)[:, n_q + n_kv:]
    cos_sin = torch.zeros(int(positions.max()) + 1, hd, device=DEV)
    ops.qk_norm_rope_kv_write(qkv.to(DEV), positions.int().to(DEV), slots.int().to(DEV), n_q, n_kv, hd, None, None, 1e-6, cos_sin, k_cache,
                              v_cache, layer)
    assert torch.equal(v_cache.cpu(), want)
