"""Expert products of small steps (csrc/kernels/moe_rows.hip) against the same equations in float64.  GPU only.

Tiles of 32 rows: one row, 16 and 17, 32 and 33 rows of an expert, all rows on two experts (several tiles of one), experts without
a row, far more experts than slots; K of one and a half units of 256 bytes; shares of the weight that are empty, partial and several passes long.  Bound: hidden
values and rows are each one bf16 rounding (2^-9) of an fp32 sum; 2-norm of the error 2^-7."""
import pytest
import torch

from test_moe_wide_gpu import _exact, _routing

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def small_experts(monkeypatch):
    """The kernel's edges are at sizes below those where it is faster."""
    from byzantine_consensus_llm_agents_amd.ops import seqmix
    monkeypatch.setattr(seqmix, "FEW_WEIGHT", 0)


@pytest.mark.parametrize("kind,limit", [("silu_gated", 0.0), ("clamped_glu", 1.5), ("relu2", 0.0)])
@pytest.mark.parametrize("routing,T,E,top,W,ff", [("even", 1, 8, 2, 64, 64), ("even", 16, 1, 1, 128, 64), ("even", 17, 1, 1, 192, 320),
                                                  ("two", 32, 4, 2, 256, 128), ("two", 33, 6, 2, 448, 192), ("even", 64, 8, 2, 2048, 2048),
                                                  ("two", 70, 8, 2, 64, 1024), ("even", 40, 40, 4, 320, 64),
                                                  ("even", 1, 64, 2, 128, 64), ("two", 3, 100, 2, 64, 64), ("even", 300, 256, 8, 1024, 1024)])
def test_few_row_experts(kind, limit, routing, T, E, top, W, ff):
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    from byzantine_consensus_llm_agents_amd.ops.seqmix import FEW_SLOTS
    assert T * top <= FEW_SLOTS * E
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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,E", [(3, 8), (40, 8), (80, 4), (300, 4)])   # position tiles of 32, 32, 64 and 256 rows (fp32: of 64)
def test_slots_without_an_expert(T, E, dtype):
    """Indices that are no expert add nothing, whatever the memory of the products held before; a token without any expert is zero."""
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops, g = get_ops("hip"), torch.Generator(device="cuda").manual_seed(T)
    bf, W, ff, top = dict(device="cuda", generator=g), 128, 128, 2
    h = torch.randn(T, W, **bf).to(dtype)
    up, down = (torch.randn(E, 2 * ff, W, **bf) * W ** -0.5).to(dtype), (torch.randn(E, W, ff, **bf) * ff ** -0.5).to(dtype)
    idx, w = _routing("even", T, E, top, g), torch.rand(T, top, **bf)
    idx[1::3, 1], idx[2::7, 0], idx[0] = -1, E, -1
    want = _exact(h, up, down, idx, w, "silu_gated", 0.0)
    for _ in range(2):
        poison = [torch.full((rows, W), float("nan"), device="cuda", dtype=dtype) for rows in (T * top, 64 * E + T * top, 256 * E + T * top)]
        del poison
        out = ops.moe_experts(h, up, down, idx, w, "silu_gated")
        assert (out[0] == 0).all() and ((out.double() - want).norm() / want.norm()).item() < 2 ** -7


@pytest.mark.parametrize("T,width,top", [(1, 1, 1), (128, 8, 2), (257, 3, 3)])
def test_table_routing(T, width, top):
    """The table's entries, also from a table and tokens that are views; a token outside the table has no expert."""
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    ops, g = get_ops("hip"), torch.Generator(device="cuda").manual_seed(T)
    table = torch.randint(0, 99, (50, 2 * width), device="cuda", generator=g, dtype=torch.int32)[:, :width]
    tokens = torch.randint(0, 50, (2 * T,), device="cuda", generator=g, dtype=torch.int32)[::2]
    idx, w = ops.moe_table_route(tokens, table, top)
    assert torch.equal(idx, table[tokens.long(), :top]) and (w == 1.0 / top).all() and w.shape == (T, top)
    assert (ops.moe_table_route(torch.tensor([-1, 50], dtype=torch.int32, device="cuda"), table, top)[0] == -1).all()
