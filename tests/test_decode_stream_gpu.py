"""Decode steps of more items than workgroups (csrc/kernels/attention.hip, decode_stream): ranges of chunks that start and end anywhere in rows and kv heads,
against the reference in float32.  GPU only."""
import random

import pytest
import torch

from byzantine_consensus_llm_agents_amd.engine.cascade import CascadeTables, plan_groups
from byzantine_consensus_llm_agents_amd.ops import reference as R

pytestmark = pytest.mark.gpu
PARTS_END = 0x7fc0e4d1   # csrc/kernels/attention.hip


@pytest.fixture(scope="module")
def ops():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    return get_ops("hip")


def _case(lens, n_kv, seed, shared=0, max_blocks=None):
    """Caches, tables and lengths; the first `shared` blocks of all rows are the same."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    rng = random.Random(seed)
    blocks = [max(1, -(-n // 16)) for n in lens]
    NB = sum(blocks) + shared + 1
    perm = list(range(1, NB))
    rng.shuffle(perm)
    head, at = perm[:shared], shared
    tables = torch.zeros(len(lens), max_blocks or max(blocks) + 3, dtype=torch.int32)
    for b, n in enumerate(blocks):
        row = (head + perm[at:at + n])[:n] if shared else perm[at:at + n]
        tables[b, :n] = torch.tensor(row, dtype=torch.int32)
        at += n
    k = torch.randn(1, NB, n_kv, 16, 128, device="cuda", generator=g).bfloat16()
    v = torch.randn(1, NB, n_kv, 128, 16, device="cuda", generator=g).bfloat16()
    v[:, 0], k[:, 0] = float("nan"), float("nan")   # nobody's page
    return k, v, tables.cuda(), torch.tensor(lens, dtype=torch.int32, device="cuda")


def _check(ops, q, k, v, tables, seq, *more):
    B = q.shape[0]
    ref = R.paged_attention(q, k, v, 0, tables, torch.arange(B + 1, dtype=torch.int32, device="cuda"), seq, 128 ** -0.5)
    out = ops.paged_attention_decode(q, k, v, 0, tables, seq, 128 ** -0.5, *more)
    torch.testing.assert_close(out.float(), ref.float(), atol=2e-2, rtol=2e-2)   # (as the other decode tests: P in bf16, one rounding of the result)
    return out


def _marks(ops, ws, B, n_q, max_blocks, cascade=False):
    """[B, n_q] how many parts the merge found behind the shared slots' end, from the marks that the attention left; -1 without one."""
    slots = ops.library.bcg_decode_max_splits(max_blocks * 16, int(cascade))
    m = ws[B * n_q * slots * 128:][:B * n_q * slots * 2].view(torch.int32).view(B, n_q, slots, 2)[..., 0]
    at = (m == PARTS_END).to(torch.int32)
    return torch.where(at.any(-1), at.argmax(-1), torch.full_like(at[..., 0], -1).to(torch.int64))


# workspaces that hold anything: NaN, marks of an end in every slot, the parts of a batch with other lengths.  Items (one round of them) and streamed ranges;
# rows without tokens; rows at the edges of a split
@pytest.mark.parametrize("lens", [[0, 1, 255, 256, 257, 30, 0, 12] * 4, [0, 1, 255, 256, 257, 1900, 700, 0] * 8], ids=["items", "streamed"])
def test_merge_takes_this_calls_parts(ops, lens):
    n_kv, G, B = 8, 5, len(lens)
    k, v, tables, seq = _case(lens, n_kv, 5)
    q = torch.randn(B, G * n_kv, 128, device="cuda").bfloat16()
    keep = seq > 0
    ref = R.paged_attention(q[keep], k, v, 0, tables[keep].contiguous(), torch.arange(int(keep.sum()) + 1, dtype=torch.int32, device="cuda"), seq[keep],
                            128 ** -0.5)
    n = ops.decode_workspace_numel(B, G * n_kv, 128, tables.shape[1], cascade=False)
    fills = [torch.full((n,), x, dtype=torch.int32, device="cuda").view(torch.float32) for x in (0x7fc00000, PARTS_END)]
    other = torch.empty(n, device="cuda")
    ops.paged_attention_decode(q, k, v, 0, tables, seq.flip(0).clamp(max=200), 128 ** -0.5, other)
    outs = [ops.paged_attention_decode(q, k, v, 0, tables, seq, 128 ** -0.5, ws) for ws in (*fills, other)]
    torch.testing.assert_close(outs[0][keep].float(), ref.float(), atol=2e-2, rtol=2e-2)
    assert not outs[0][~keep].any() and all(torch.equal(outs[0], o) for o in outs[1:])
    parts, items = _marks(ops, fills[0], B, G * n_kv, tables.shape[1]), (seq + 255) // 256
    assert torch.equal(parts, items[:, None].expand_as(parts).where(keep[:, None], torch.full_like(parts, -1))) == (int(items.sum()) * n_kv <= 512)


# 1 to 8 query heads a kv head; rows of one token, one chunk, one split and their neighbours, rows without tokens at the ends and between; all rows equal
# (ranges that end with a pair); one long row among short ones (ranges longer than their share); a table as long as its longest row
@pytest.mark.parametrize("G", [1, 4, 5, 8])
@pytest.mark.parametrize("kind", ["edges", "equal", "one long", "random"])
def test_ranges(ops, kind, G):
    rng = random.Random(G)
    n_kv, B = 8, 97
    lens = {"edges": [rng.choice([0, 1, 16, 31, 32, 33, 255, 256, 257, 300, 511]) for _ in range(B)], "equal": [288] * B,
            "one long": [4000] + [rng.randint(257, 400) for _ in range(B - 1)], "random": [rng.randint(1, 900) for _ in range(B)]}[kind]
    if kind == "edges":
        lens[0] = lens[1] = lens[-1] = 0
    k, v, tables, seq = _case(lens, n_kv, G)
    q = torch.randn(B, G * n_kv, 128, device="cuda").bfloat16()
    keep = seq > 0
    B_, t = int(keep.sum()), tables
    ref = R.paged_attention(q[keep], k, v, 0, t[keep].contiguous(), torch.arange(B_ + 1, dtype=torch.int32, device="cuda"), seq[keep], 128 ** -0.5)
    out = ops.paged_attention_decode(q, k, v, 0, t, seq, 128 ** -0.5)
    torch.testing.assert_close(out[keep].float(), ref.float(), atol=2e-2, rtol=2e-2)
    assert not out[~keep].any()                 # a row without tokens is zeros, as from the items
    assert int(((seq + 255) // 256).sum()) * n_kv > 512   # (more than a round of items)
    assert torch.equal(out, ops.paged_attention_decode(q, k, v, 0, t, seq, 128 ** -0.5))


def _streamed(ops, q, k, v, tables, seq, cascade=None):
    """The call's result; its parts are not the items': the step was streamed."""
    B, n_q, _ = q.shape
    ws = torch.full((ops.decode_workspace_numel(B, n_q, 128, tables.shape[1], cascade=cascade is not None),), float("nan"), device="cuda")
    out = _check(ops, q, k, v, tables, seq, ws, cascade)
    parts = _marks(ops, ws, B, n_q, tables.shape[1], cascade is not None)
    begin = 0 if cascade is None else cascade.kv_begin[:B]
    base = 0 if cascade is None else cascade.split_base[:B, None]
    items = (seq - begin + 255) // 256
    assert int(items.sum()) * k.shape[2] > 512
    assert not torch.equal(parts - base, items[:, None].expand_as(parts))
    return out


def test_most_rows_and_longest_context(ops):
    """As many rows as a call takes, and contexts of the most slots (no slot to spare: the ranges are so long that a row's parts fit) among short ones."""
    rng = random.Random(1)
    k, v, tables, seq = _case([rng.randint(1, 70) for _ in range(2048)], 2, 1)
    _streamed(ops, torch.randn(2048, 8, 128, device="cuda").bfloat16(), k, v, tables, seq)
    limit = ops.decode_max_context(False)
    assert ops.library.bcg_decode_max_splits(limit, 0) == 64
    for lens in ([limit] + [rng.randint(1, 300) for _ in range(700)], [limit, limit - 1, 5, limit - 255] * 3 + [rng.randint(1, 300) for _ in range(300)]):
        k, v, tables, seq = _case(lens, 1, 2, max_blocks=limit // 16)
        _streamed(ops, torch.randn(len(lens), 5, 128, device="cuda").bfloat16(), k, v, tables, seq)


def test_longest_context_behind_shared_prefixes(ops):
    """The slots of the shared pass taken, the own ones at their limit."""
    rng = random.Random(4)
    n_kv, G, shared, limit = 2, 5, 23, ops.decode_max_context(True)
    assert ops.library.bcg_decode_max_splits(limit, 1) == 64
    lens = [limit, limit - 100] + [shared * 16 + rng.randint(1, 600) for _ in range(250)]
    k, v, tables, seq = _case(lens, n_kv, 3, shared, max_blocks=limit // 16)
    t = CascadeTables(len(lens), "cuda")
    t.upload(plan_groups([(i, tables[i, :-(-n // 16)].tolist()) for i, n in enumerate(lens)]), heads_per_kv=G)
    assert int(t.split_base[0]) > 0
    _streamed(ops, torch.randn(len(lens), G * n_kv, 128, device="cuda").bfloat16(), k, v, tables, seq, t)


def test_behind_shared_prefixes_and_replayed(ops):
    """The rows' own tokens behind a shared prefix, in a captured step whose lengths grow between replays."""
    n_kv, G, B, shared = 8, 5, 150, 23
    lens = [shared * 16 + 200 + 7 * (i % 60) for i in range(B)]
    k, v, tables, seq = _case([n + 8 for n in lens], n_kv, 3, shared)
    seq -= 8
    q = torch.randn(B, G * n_kv, 128, device="cuda").bfloat16()
    t = CascadeTables(B, "cuda")
    t.upload(plan_groups([(i, tables[i, :-(-n // 16)].tolist()) for i, n in enumerate(lens)]), heads_per_kv=G)
    _streamed(ops, q, k, v, tables, seq, t)
    ws = torch.empty(ops.decode_workspace_numel(B, G * n_kv, 128, tables.shape[1]), dtype=torch.float32, device="cuda")
    args = (q, k, v, 0, tables, seq, 128 ** -0.5, ws)
    ops.paged_attention_decode(*args)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.paged_attention_decode(*args)
    for _ in range(3):
        seq += 2
        want = _check(ops, q, k, v, tables, seq)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
