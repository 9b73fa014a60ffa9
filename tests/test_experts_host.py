"""Expert layers of the HIP backend where no kernel runs: routing by token id of host tensors, wrapped tensors and traces is a gather, as
in the reference; a step without tokens or without chosen experts is zeros.  No GPU."""
import os

import pytest
import torch

from byzantine_consensus_llm_agents_amd.ops import reference


@pytest.fixture(scope="module")
def ops():
    from byzantine_consensus_llm_agents_amd.ops.hip import hip_ops
    from byzantine_consensus_llm_agents_amd.utils.build import kernels_target
    if not os.path.exists(kernels_target()):
        pytest.skip("kernel library not built")
    return hip_ops()


@pytest.mark.parametrize("T,width,top", [(1, 1, 1), (70, 8, 2), (5, 3, 3), (0, 4, 2)])
def test_host_tensors(ops, T, width, top):
    g = torch.Generator().manual_seed(T)
    for table in (torch.randint(0, 99, (50, width), generator=g, dtype=torch.int32), torch.randint(0, 99, (50, 2 * width), generator=g, dtype=torch.int32)[:, ::2]):
        tokens = torch.randint(0, 50, (T,), generator=g, dtype=torch.int32)
        idx, w = ops.moe_table_route(tokens, table, top)
        want, ww = reference.moe_table_route(tokens, table, top)
        assert torch.equal(idx, want) and torch.equal(w, ww) and idx.dtype == torch.int32 and idx.shape == w.shape == (T, top)
    with pytest.raises((IndexError, RuntimeError)):
        ops.moe_table_route(torch.tensor([50], dtype=torch.int32), table, top)


def test_batched_by_a_transform(ops):
    table = torch.arange(60, dtype=torch.int32).view(20, 3)
    tokens = torch.tensor([[0, 19, 3], [7, 7, 1]], dtype=torch.int32)
    assert torch.equal(torch.func.vmap(lambda t: ops.moe_table_route(t, table, 2)[0])(tokens), table[tokens.long(), :2])


@pytest.mark.parametrize("T,top", [(0, 2), (3, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_no_slots(ops, T, top, dtype):
    h, up, down = torch.ones(T, 64, dtype=dtype), torch.ones(4, 128, 64, dtype=dtype), torch.ones(4, 64, 64, dtype=dtype)
    idx, w = torch.zeros(T, top, dtype=torch.int32), torch.zeros(T, top)
    out = ops.moe_experts(h, up, down, idx, w, "silu_gated")
    assert torch.equal(out, reference.moe_experts(h, up, down, idx, w, "silu_gated")) and out.shape == (T, 64) and out.dtype == torch.float32
