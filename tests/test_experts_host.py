"""Expert layers of the HIP backend where no kernel runs: routing by token id of host tensors, wrapped tensors and traces is a gather, as
in the reference; a step without tokens or without chosen experts is zeros.  No GPU."""
import os
import random

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


def test_tiles_of_few_rows():
    """The rule for position tiles of 32 rows: never past its limits, and what it counts is enough for the tiles that hold slots."""
    from byzantine_consensus_llm_agents_amd.ops.seqmix import FEW_SLOTS, few_row_tiles
    rng, over, taken = random.Random(5), 0, 0
    for _ in range(400):
        E, top = rng.choice([1, 2, 8, 31, 64, 200, 256]), rng.choice([1, 2, 8])
        n = rng.randint(1, max(1, FEW_SLOTS * E // top)) * top
        held = few_row_tiles(n, E, 2048, 1024, 32)
        if n > FEW_SLOTS * E or held == 0:
            continue
        counts = [0] * E
        for _ in range(n):
            counts[rng.randrange(E)] += 1
        tiles = sum(-(-c // 32) for c in counts)
        assert tiles <= (n + min(E, n) * 31) // 32      # what is launched
        taken, over = taken + 1, over + (tiles > held + 1 + E // 30)
    assert taken > 200 and over < 0.06 * taken           # two standard deviations
    assert few_row_tiles(24 * 8 + 1, 8, 2048, 2048, 32) == 0 and few_row_tiles(128, 8, 2048, 2048, 32) == 8
    assert few_row_tiles(128, 128, 2048, 1024, 32) == 0 and few_row_tiles(2048, 256, 1024, 256, 32) == 0
    assert few_row_tiles(1, 256, 4096, 3072, 32) == 1 and few_row_tiles(16, 8, 512, 256, 32) == 0
