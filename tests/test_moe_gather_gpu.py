"""Rows gathered by the expert product itself (bcg_gemm_w4_grouped): more tiles than CUs, so that workgroups go on to tiles of other rows, with one to eight
steps of K per tile.  Against float64, the bound of the other wide expert tests; a second call on other rows must not see the first one's."""
import pytest
import torch

from test_moe_wide_gpu import _exact, _routing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,limit", [("silu_gated", 0.0), ("relu2", 0.0)])
@pytest.mark.parametrize("T,E,top,W,ff", [(6001, 4, 2, 64, 1024), (9000, 7, 1, 128, 1024), (3000, 5, 3, 512, 1280)])
def test_gathered_rows(kind, limit, T, E, top, W, ff):
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops, g = get_ops("hip"), torch.Generator(device="cuda").manual_seed(T)
    bf = dict(device="cuda", generator=g)
    n_up = 2 * ff
    if kind == "relu2":
        ff = n_up
    assert (T * top // 256) * (n_up // 256) > torch.cuda.get_device_properties(0).multi_processor_count
    up, down = (torch.randn(E, n_up, W, **bf) * W ** -0.5).bfloat16(), (torch.randn(E, W, ff, **bf) * ff ** -0.5).bfloat16()
    for _ in range(2):
        h, idx, w = torch.randn(T, W, **bf).bfloat16(), _routing("even", T, E, top, g), torch.rand(T, top, **bf)
        idx[5] = -1   # (a token without an expert)
        want = _exact(h, up, down, idx, w, kind, limit)
        out = ops.moe_experts(h, up, down, idx, w, kind, limit)
        assert ((out.double() - want).norm() / want.norm()).item() < 2 ** -7
