"""Rotary embedding, cache write and attention of a decode step in one launch (csrc/kernels/attention.hip, decode_pair_kernel), heads of 64, against the
separate operations.  GPU only.

Both round queries and keys to bf16 after the same fp32 arithmetic and store the same bytes (a root mean square summed in
another order can move a key by one rounding); the outputs differ by fp32 summation order before one bf16 rounding: 2^-8 of
their size, and 2^-7 where a rounding of a query falls the other way."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# contexts at the edges of pages (16), chunks (32), waves (64) and splits (256); 0: a row without tokens
LENS = [1, 15, 16, 17, 31, 32, 33, 64, 65, 255, 256, 257, 320, 511, 512, 513, 1100, 2049, 0]


@pytest.fixture(scope="module")
def ops():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    return get_ops("hip")


def _case(lens, n_q, n_kv, hd, norm, seed=0, parked=()):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dev, B = "cuda", len(lens)
    width = max(1, max(-(-n // 16) for n in lens))
    blocks = B * width + 2
    order = torch.randperm(blocks - 1, generator=torch.Generator().manual_seed(seed)) + 1
    table = order[:B * width].view(B, width).to(torch.int32)
    k = torch.randn(2, blocks, n_kv, 16, hd, device=dev, generator=g).to(torch.bfloat16)
    v = torch.randn(2, blocks, n_kv, hd, 16, device=dev, generator=g).to(torch.bfloat16)
    slots, pos = [], []
    for b, n in enumerate(lens):
        p = max(n - 1, 0)
        pos.append(p)
        slots.append(0 if n == 0 or b in parked else int(table[b, p // 16]) * 16 + p % 16)
        if n and b not in parked:     # whatever was there before, never to be seen
            k[1, slots[-1] // 16, :, slots[-1] % 16] = float("nan")
            v[1, slots[-1] // 16, :, :, slots[-1] % 16] = float("inf")
    i32 = dict(dtype=torch.int32, device=dev)
    qkv = torch.randn(B, (n_q + 2 * n_kv) * hd, device=dev, generator=g).to(torch.bfloat16)
    nw = [(1 + 0.2 * torch.randn(hd, device=dev, generator=g)).to(torch.bfloat16) if norm else None for _ in range(2)]
    ang = torch.rand(max(4096, *lens), hd // 2, device=dev, generator=g) * 6.28   # (a row for every position)
    return dict(qkv=qkv, positions=torch.tensor(pos, **i32), slots=torch.tensor(slots, **i32), n_q=n_q, n_kv=n_kv, hd=hd, q_norm=nw[0],
                k_norm=nw[1], eps=1e-6, cos_sin=torch.cat([ang.cos(), ang.sin()], 1).contiguous()), k, v, table.to(dev), torch.tensor(lens, **i32)


def _separate(ops, c, k, v, table, lens):
    q = ops.qk_norm_rope_kv_write(c["qkv"], c["positions"], c["slots"], c["n_q"], c["n_kv"], c["hd"], c["q_norm"], c["k_norm"],
                                  c["eps"], c["cos_sin"], k, v, 1, contiguous=False)
    return ops.paged_attention_decode(q, k, v, 1, table, lens, c["hd"] ** -0.5)


def _fused(ops, c, k, v, table, lens):
    return ops.decode_attention_pairs(c["qkv"], c["positions"], c["slots"], c["n_q"], c["n_kv"], c["hd"], c["q_norm"], c["k_norm"], c["eps"],
                                c["cos_sin"], k, v, 1, table, lens, c["hd"] ** -0.5)


def _same_cache(c, k0, v0, k, v, k1, v1, norm, rows=None):
    """The entries that a step stored (layer 1 at the rows' slots; `rows`: of these rows), one by one: V and keys without a norm the
    same bits, normalised keys one rounding apart at most (neighbouring bf16 values are up to 2^-7 apart; 2^-18: fp32 sums of two
    products of up to 8 that cancel).  All other bits of both caches are untouched."""
    every = c["slots"].long()
    at = every if rows is None else every[rows]
    page, off = at // 16, at % 16
    ks, kf = k[1, page, :, off].float(), k1[1, page, :, off].float()
    assert torch.isfinite(kf).all()
    assert bool(((kf - ks).abs() <= 2 ** -7 * ks.abs() + 2 ** -18).all()) if norm else torch.equal(kf, ks)
    assert torch.equal(v1[1, page, :, :, off], v[1, page, :, :, off])
    for now, was, entry in ((k1, k0, (1, every // 16, slice(None), every % 16)), (v1, v0, (1, every // 16, slice(None), slice(None), every % 16))):
        rest = now.clone()
        rest[entry] = was[entry]
        assert torch.equal(rest.view(torch.int16), was.view(torch.int16))


@pytest.mark.parametrize("n_q,n_kv,norm", [(14, 2, False), (40, 8, True), (16, 1, False), (4, 4, True)])
def test_against_separate_operations(ops, n_q, n_kv, norm):
    c, k, v, table, lens = _case(LENS, n_q, n_kv, 64, norm, seed=n_q)
    (k0, v0), (k1, v1) = (k.clone(), v.clone()), (k.clone(), v.clone())
    want = _separate(ops, c, k, v, table, lens)
    got = _fused(ops, c, k1, v1, table, lens)
    _same_cache(c, k0, v0, k, v, k1, v1, norm)
    assert torch.isfinite(got).all() and (got[-1] == 0).all()
    for b in range(len(LENS) - 1):
        off = ((got[b].double() - want[b].double()).norm() / want[b].double().norm()).item()
        assert off < 2 ** -7, (LENS[b], off)


def test_parked_rows_and_graph_replays(ops):
    """A row whose slot is not its newest position reads the cache as it is."""
    lens = [1, 300, 700, 1, 513]
    c, k, v, table, sl = _case(lens, 10, 2, 64, True, seed=3, parked=(0, 2))
    (k0, v0), (k1, v1) = (k.clone(), v.clone()), (k.clone(), v.clone())
    want = _separate(ops, c, k, v, table, sl)
    _fused(ops, c, k1, v1, table, sl)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = _fused(ops, c, k1, v1, table, sl)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert ((out.double() - want.double()).norm() / want.double().norm()).item() < 2 ** -7
        _same_cache(c, k0, v0, k, v, k1, v1, True, rows=[1, 3, 4])


def test_strided_caches_are_refused(ops):
    """Caches that are views of larger ones: an error before any launch, as from the separate operations."""
    c, k, v, table, sl = _case([5, 40], 4, 2, 64, False, seed=1)
    f8 = torch.float8_e4m3fn
    for bad in ((k.repeat(2, 1, 1, 1, 1)[::2], v), (k, v.repeat(2, 1, 1, 1, 1)[::2]), (k.to(f8), v.to(f8))):
        before = [t.float().nan_to_num() for t in bad]
        for call in (_separate, _fused)[bad[0].dtype == f8:]:   # (fp8 caches are the separate operations' alone)
            with pytest.raises(ValueError):
                call(ops, c, *bad, table, sl)
        assert all(torch.equal(t.float().nan_to_num(), b) for t, b in zip(bad, before))
