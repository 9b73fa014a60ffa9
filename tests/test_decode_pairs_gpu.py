"""A decode step's attention by a workgroup for each part of a (row, kv head) pair (csrc/kernels/attention.hip, decode_pair_kernel) against rotary
launch, items or stream, and merge.  GPU only.

Bounds as in test_decode_fused_gpu.py: the same bytes are stored, outputs differ by fp32 summation order before one bf16 rounding."""
import pytest
import torch

from test_decode_fused_gpu import _case, _same_cache, _separate, ops  # noqa: F401

pytestmark = pytest.mark.gpu

# contexts at the edges of pages (16), chunks (32) and turns of 2, 4 and 8 waves (64, 128, 256); 0: a row without tokens
LENS = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 256, 257, 300, 511, 513, 1100, 2049, 0]


def _pairs(ops, c, k, v, table, lens, parts=None, workspace=None):
    return ops.decode_attention_pairs(c["qkv"], c["positions"], c["slots"], c["n_q"], c["n_kv"], c["hd"], c["q_norm"], c["k_norm"], c["eps"],
                                      c["cos_sin"], k, v, 1, table, lens, c["hd"] ** -0.5, workspace, parts)


# times: the lengths repeated (but 0: rows without tokens store to one slot), so that the pairs are past the line from which on workgroups have fewer waves
@pytest.mark.parametrize("n_q,n_kv,hd,norm,parts,times", [
    (14, 2, 64, False, 1, 1), (16, 1, 64, True, 3, 1), (4, 4, 64, True, 1, 7), (14, 2, 64, False, 5, 3), (4, 4, 64, False, None, 1),
    (40, 8, 128, True, 1, 1), (16, 1, 128, False, 2, 1), (48, 8, 128, False, 7, 1), (32, 8, 128, True, 1, 7), (5, 1, 128, True, 64, 1), (6, 1, 128, True, None, 1)])
def test_against_separate_operations(ops, n_q, n_kv, hd, norm, parts, times):
    c, k, v, table, lens = _case(LENS[:-1] * times + [0], n_q, n_kv, hd, norm, seed=n_q + hd)
    (k0, v0), (k1, v1) = (k.clone(), v.clone()), (k.clone(), v.clone())
    want = _separate(ops, c, k, v, table, lens)
    got = _pairs(ops, c, k1, v1, table, lens, parts)
    _same_cache(c, k0, v0, k, v, k1, v1, norm)
    assert torch.isfinite(got).all() and (got[lens == 0] == 0).all()
    live = lens > 0
    off = (got[live].double() - want[live].double()).norm(dim=1) / want[live].double().norm(dim=1)
    assert bool((off < 2 ** -7).all()), off.max()


@pytest.mark.parametrize("parts", [1, 4])
def test_wide_tables_parked_rows_and_graph_replays(ops, parts):
    """A table with room behind every context, whose entries there are no pages; parts without a chunk; a row whose slot is not its newest position."""
    c, k, v, table, sl = _case([1, 300, 700, 1, 513], 10, 2, 128, True, seed=3, parked=(0, 2))
    used = torch.arange(table.shape[1], device="cuda")[None] * 16 < sl[:, None]
    table = torch.cat([torch.where(used, table, 1 << 28), torch.full((5, 300), 1 << 28, dtype=torch.int32, device="cuda")], 1).contiguous()
    (k0, v0), (k1, v1) = (k.clone(), v.clone()), (k.clone(), v.clone())
    want = _separate(ops, c, k, v, table, sl)
    ws = torch.full((5 * 10 * parts * 130,), float("nan"), device="cuda")
    _pairs(ops, c, k1, v1, table, sl, parts, ws)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = _pairs(ops, c, k1, v1, table, sl, parts, ws)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert ((out.double() - want.double()).norm() / want.double().norm()).item() < 2 ** -7
        _same_cache(c, k0, v0, k, v, k1, v1, True, rows=[1, 3, 4])
