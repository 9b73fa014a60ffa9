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


def _float64(c, k, v, table, lens):
    """The attention in float64 over what the separate operations rotated and stored."""
    q = _rotated(c)
    out = []
    for b, n in enumerate(lens.tolist()):
        pages = table[b, :-(-n // 16)].long()
        kk = k[1, pages].permute(1, 0, 2, 3).reshape(c["n_kv"], -1, c["hd"])[:, :n].double()
        vv = v[1, pages].permute(1, 0, 3, 2).reshape(c["n_kv"], -1, c["hd"])[:, :n].double()
        g = c["n_q"] // c["n_kv"]
        s = torch.softmax(torch.matmul(q[b].view(c["n_kv"], g, c["hd"]), kk.transpose(1, 2).contiguous()) * c["hd"] ** -0.5, -1)
        out.append(torch.matmul(s, vv).reshape(-1))
    return torch.stack(out)


def _rotated(c):
    x = c["qkv"].double().view(c["qkv"].shape[0], -1, c["hd"])[:, :c["n_q"]]
    if c["q_norm"] is not None:
        x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + c["eps"]) * c["q_norm"].double()
    cs = c["cos_sin"][c["positions"].long()].double()[:, None]
    h = c["hd"] // 2
    cos, sin, a, b = cs[..., :h], cs[..., h:], x[..., :h], x[..., h:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1).to(torch.bfloat16).double()


def _cut(lens, pairs_per_row, rule):
    """Parts of every row, as find_share of csrc/kernels/common.h has them."""
    parts, one, each, ways, _ = rule
    chunks = (lens.cpu() + 31) // 32
    share = chunks * ways / (int(chunks.sum()) * pairs_per_row)
    return torch.where(chunks > one, torch.minimum(share.long(), (chunks + each - 1) // each).clamp(1, parts), 1)


# long rows beside short ones, few and many pairs, up to the most parts, in tables as wide as they need and wider; (40 rows: the range of pairs that are cut finer)
@pytest.mark.parametrize("n_q,n_kv,hd,lens,room", [
    (40, 8, 128, [7000] + [300] * 9, 0), (40, 8, 128, [60] * 20 + [5000] + [90] * 14, 512), (14, 2, 64, [4000, 30, 9000], 0), (10, 2, 128, [3000] * 3, 0),
    (32, 8, 128, [100] * 130 + [8000], 0), (14, 2, 64, [2500], 512), (40, 8, 128, [1500] * 40, 0)])
def test_rows_cut_by_the_rule(ops, n_q, n_kv, hd, lens, room):
    """Outputs in float64's, the parts that the rule says (and no others) in the workspace, on two streams the same bits."""
    from byzantine_consensus_llm_agents_amd.ops.hip import part_rule
    c, k, v, table, sl = _case(lens, n_q, n_kv, hd, True, seed=n_q)
    if room > table.shape[1]:
        table = torch.cat([table, torch.full((len(lens), room - table.shape[1]), 1 << 28, dtype=torch.int32, device="cuda")], 1).contiguous()
    rule = part_rule(len(lens) * n_kv, 128 * hd, -(-table.shape[1] // 2))
    cut = _cut(sl, n_kv, rule)
    assert cut.max() > 1 and int((cut - 1).sum()) * n_kv <= rule[4]
    G, extra = n_q // n_kv, rule[4]
    ws = torch.full((2 * extra * G * (hd + 2),), float("nan"), device="cuda")
    got = _pairs(ops, c, k, v, table, sl, None, ws)
    used = (~torch.isnan(ws[:2 * extra * G * hd].view(2 * extra, -1))).all(1)
    assert int(used[:extra].sum()) == int((cut - 1).sum()) * n_kv and int(used[extra:].sum()) == int((cut > 1).sum()) * n_kv
    want = _float64(c, k, v, table, sl)
    off = (got.double() - want).view(len(lens), n_q, hd).norm(dim=-1) / want.view(len(lens), n_q, hd).norm(dim=-1)
    assert bool((off < 2 ** -7).all()), off.max()
    streams, outs = [torch.cuda.Stream() for _ in range(2)], [[], []]
    torch.cuda.synchronize()
    for _ in range(4):
        for s, o in zip(streams, outs):
            with torch.cuda.stream(s):
                o.append(_pairs(ops, c, k, v, table, sl))
    torch.cuda.synchronize()
    assert all(torch.equal(t, got) for o in outs for t in o)


def test_short_rows_in_wide_tables_stay_whole(ops):
    c, k, v, table, sl = _case([500, 300, 800, 40], 14, 2, 64, False, seed=1)
    narrow = _pairs(ops, c, k, v, table, sl)
    wide = torch.cat([table, torch.full((4, 1000 - table.shape[1]), 1 << 28, dtype=torch.int32, device="cuda")], 1).contiguous()
    ws = torch.full((1 << 18,), float("nan"), device="cuda")
    assert torch.equal(_pairs(ops, c, k, v, wide, sl, None, ws), narrow) and torch.isnan(ws).all()
