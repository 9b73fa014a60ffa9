"""Single-token rows of exact head sizes by a workgroup per (row, KV head) pair (csrc/kernels/seqmix_attention.hip, decode_pair_kernel) against the
float32 reference.  GPU only.

bf16 operands, fp32 sums; probabilities and outputs are rounded to bf16 (2^-9 each) before and after sums over keys of both signs: a head's output is
off by 2^-8 of its own norm, 2^-7 where the maps nearly cancel.  (A chunk of 32 keys left out of 1025 is off by 2^-3.)"""
import pytest
import torch

from byzantine_consensus_llm_agents_amd.models.transformer import AttnMeta
from byzantine_consensus_llm_agents_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"
# contexts at the edges of pages (16), chunks (32) and turns of 2 and 4 waves (64, 128)
LENS = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 300, 513, 1025]
KINDS = {"plain": {}, "window": dict(window=37), "long window": dict(window=300), "chunk": dict(chunk=50), "keep": dict(window=40, keep=5), "keep far": dict(window=70, keep=140),
         "sink": dict(sink=True, window=100), "far sink": dict(sink=True, window=700), "shaped": dict(softcap=3.0, slopes=True), "shaped window": dict(softcap=3.0, slopes=True, window=100)}


@pytest.fixture(scope="module")
def ops():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    return get_ops("hip")


def _case(H, G, maps, dim, vdim, kind, rows, wide, eps, seed, lens=None):
    lens = lens or (LENS * rows)[:rows]
    g = torch.Generator(device=DEV).manual_seed(seed)
    per = [-(-n // 16) for n in lens]
    blocks = sum(per) + 1
    ids = torch.randperm(blocks - 1, generator=torch.Generator().manual_seed(seed)) + 1
    bt, at = torch.full((rows, max(per) + wide), 1 << 28, dtype=torch.int32), 0   # (no pages behind the contexts)
    for b, n in enumerate(per):
        bt[b, :n] = ids[at:at + n].to(torch.int32)
        at += n
    k = torch.randn(blocks, G, 16, maps * dim, device=DEV, generator=g).to(torch.bfloat16)
    v = torch.randn(blocks, G, vdim, 16, device=DEV, generator=g).to(torch.bfloat16)
    kw = dict(KINDS[kind])
    if kw.get("sink"):
        kw["sink"] = torch.randn(H, device=DEV, generator=g)
    if kw.get("slopes"):
        kw["slopes"] = torch.rand(H, device=DEV, generator=g) * 0.1
    q = torch.randn(rows, H, maps * dim, device=DEV, generator=g).to(torch.bfloat16)
    lens = torch.tensor(lens, dtype=torch.int32, device=DEV)
    return q, k, v, bt.to(DEV), lens, (dim ** -0.5, maps, 0.35, eps, 0.4, vdim), kw


def _close(got, want, vdim):
    got, want = (t.double().view(t.shape[0], -1, vdim) for t in (got, want))
    off = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert bool((off < 2 ** -7).all()), (off.max(), off.argmax())


# parts: of every pair; None: by the rule, which cuts the rows of 1025 keys where the pairs are few and the keys wide.  wide: pages that the table has room for besides
@pytest.mark.parametrize("H,G,maps,dim,vdim,kind,rows,wide,parts,eps", [
    (32, 8, 2, 64, 128, "plain", 16, 0, None, 1e-5), (16, 4, 2, 64, 128, "plain", 16, 900, None, 1e-5), (16, 16, 2, 32, 32, "plain", 80, 0, None, 1e-5),
    (6, 2, 2, 48, 96, "plain", 16, 0, None, -1.0), (40, 1, 1, 192, 128, "window", 16, 0, None, -1.0), (4, 2, 1, 96, 64, "plain", 16, 0, None, 1e-5),
    (8, 4, 1, 128, 128, "keep", 16, 0, None, -1.0), (8, 4, 1, 64, 64, "keep far", 16, 900, None, -1.0), (64, 64, 1, 128, 128, "keep", 20, 0, None, 1e-5),
    (4, 2, 1, 64, 128, "chunk", 16, 0, None, 1e-5), (4, 2, 1, 128, 128, "sink", 16, 0, None, -1.0), (4, 2, 1, 192, 192, "shaped", 16, 0, None, -1.0),
    (4, 2, 1, 256, 256, "plain", 16, 0, None, -1.0), (4, 2, 1, 256, 256, "shaped", 600, 0, None, -1.0), (16, 16, 1, 192, 128, "plain", 70, 0, None, -1.0),
    # cut: every mask and the sink over two, some and the most parts, parts without a chunk, several column groups, two waves
    (32, 8, 2, 64, 128, "plain", 16, 0, 2, 1e-5), (16, 4, 2, 64, 128, "plain", 16, 0, 16, -1.0), (40, 1, 1, 192, 128, "long window", 16, 40, 5, -1.0),
    (17, 1, 1, 192, 128, "plain", 16, 0, 16, -1.0), (8, 4, 1, 128, 128, "keep", 16, 0, 2, -1.0), (8, 4, 1, 64, 64, "keep far", 16, 40, 5, 1e-5),
    (4, 2, 1, 128, 128, "keep far", 16, 0, 16, -1.0), (4, 2, 1, 64, 128, "chunk", 16, 0, 2, 1e-5), (4, 2, 1, 128, 128, "far sink", 16, 0, 5, -1.0),
    (4, 1, 1, 128, 128, "far sink", 16, 0, 16, 1e-5), (4, 2, 1, 192, 192, "shaped", 16, 0, 5, -1.0), (4, 2, 1, 256, 256, "shaped", 16, 0, 16, -1.0),
    (8, 4, 2, 32, 32, "plain", 160, 0, 3, 1e-5), (6, 2, 2, 48, 96, "plain", 16, 0, 7, 1e-5)])
def test_against_reference(ops, H, G, maps, dim, vdim, kind, rows, wide, parts, eps):
    q, k, v, bt, lens, args, kw = _case(H, G, maps, dim, vdim, kind, rows, wide, eps, seed=dim + rows)
    assert ops.library.bcg_multimap_pairs(maps, dim, vdim, int(kind == "shaped"), kw.get("keep", 0))
    kp, vp = ops.kv_from_logical(k, v)
    got = ops.multimap_attention(q, kp, vp, AttnMeta(positions=None, slots=None, block_tables=bt, seq_lens=lens, decode=True), *args, **kw, parts=parts)
    want = ref.multimap_attention(q, k, v, bt, torch.arange(rows + 1, dtype=torch.int32, device=DEV), lens, *args, **kw)
    _close(got, want, vdim)


def test_long_rows_beside_short_ones(ops):
    """By the rule: rows of 5000 and 3000 keys among short ones are cut, also in a table with room for 16384, on two streams at once."""
    lens = [40, 5000, 33, 3000] + [50] * 60
    q, k, v, bt, sl, args, _ = _case(8, 2, 2, 64, 128, "plain", len(lens), 800, 1e-5, seed=5, lens=lens)
    kp, vp = ops.kv_from_logical(k, v)
    meta = AttnMeta(positions=None, slots=None, block_tables=bt, seq_lens=sl, decode=True)
    want = ref.multimap_attention(q, k, v, bt, torch.arange(len(lens) + 1, dtype=torch.int32, device=DEV), sl, *args)
    first = ops.multimap_attention(q, kp, vp, meta, *args)
    _close(first, want, 128)
    streams, outs = [torch.cuda.Stream() for _ in range(2)], [[], []]
    torch.cuda.synchronize()
    for _ in range(5):
        for s, o in zip(streams, outs):
            with torch.cuda.stream(s):
                o.append(ops.multimap_attention(q, kp, vp, meta, *args))
    torch.cuda.synchronize()
    assert all(torch.equal(t, first) for o in outs for t in o)   # (parts are added in their order, whoever comes last)


@pytest.mark.parametrize("kind,parts", [("window", None), ("long window", None), ("long window", 5), ("chunk", None), ("keep", None), ("keep far", 2), ("shaped window", None)])
def test_pages_in_front_of_the_window(ops, kind, parts):
    """Pages wholly in front of a window (or between it and the kept keys' chunks) hold infinities and NaN: no query sees them."""
    q, k, v, bt, lens, args, kw = _case(4, 2, 1, 128, 128, kind, 16, 0, -1.0, seed=4)
    want = ref.multimap_attention(q, k, v, bt, torch.arange(17, dtype=torch.int32, device=DEV), lens, *args, **kw)
    for b, n in enumerate(lens.tolist()):
        lo = max(0, n - kw["window"]) if "window" in kw else (n - 1) - (n - 1) % kw["chunk"]
        for page in range(2 * (-(-kw.get("keep", 0) // 32)), lo // 16):
            k[bt[b, page]], v[bt[b, page]] = float("nan"), float("inf")
    kp, vp = ops.kv_from_logical(k, v)
    got = ops.multimap_attention(q, kp, vp, AttnMeta(positions=None, slots=None, block_tables=bt, seq_lens=lens, decode=True), *args, **kw, parts=parts)
    _close(got, want, 128)


def test_single_rows_and_graph_replays(ops):
    """Rows of a packed step in an order of their own, several parts, replayed."""
    q, k, v, bt, lens, args, _ = _case(16, 4, 2, 64, 128, "plain", 6, 1500, 1e-5, seed=9, lens=[300, 17, 1025, 1, 1500, 700])
    kp, vp = ops.kv_from_logical(k, v)
    order = torch.tensor([4, 0, 5, 2], device=DEV)
    single = torch.stack([order, order.flip(0)], 1).to(torch.int32).contiguous()   # row order[i] is sequence order[-1 - i]'s
    meta = AttnMeta(positions=None, slots=None, block_tables=bt, seq_lens=lens, q_start=torch.zeros(7, dtype=torch.int32, device=DEV), decode=False, tile_rows=64,
                    tiles=torch.zeros(0, 3, dtype=torch.int32, device=DEV), single=single)
    seqs = order.flip(0)
    want = ref.multimap_attention(q[order], k, v, bt[seqs], torch.arange(5, dtype=torch.int32, device=DEV), lens[seqs], *args)
    for parts in (None, 4):   # (the rule cuts the rows of 1025 and 1500 keys)
        eager = ops.multimap_attention(q, kp, vp, meta, *args, parts=parts)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            out = ops.multimap_attention(q, kp, vp, meta, *args, parts=parts)
        for _ in range(3):
            out.zero_()
            g.replay()
            _close(ops.multimap_attention(q, kp, vp, meta, *args, parts=parts)[order], want, 128)
            torch.cuda.synchronize()
            assert torch.equal(out[order], eager[order])
            _close(out[order], want, 128)


@pytest.mark.parametrize("H,G,maps,dim,vdim,kind,eps", [(8, 2, 2, 64, 128, "plain", 1e-5), (6, 2, 2, 48, 96, "plain", -1.0), (4, 2, 1, 128, 128, "window", -1.0),
                                                        (4, 2, 1, 192, 128, "plain", -1.0), (8, 4, 1, 64, 64, "keep far", 1e-5), (4, 2, 1, 256, 256, "shaped", -1.0)])
def test_caches_off_16_bytes(ops, H, G, maps, dim, vdim, kind, eps):
    """Views that begin 8 bytes into their memory take the splits."""
    q, k, v, bt, lens, args, kw = _case(H, G, maps, dim, vdim, kind, 16, 0, eps, seed=2)
    moved = []
    for t in ops.kv_from_logical(k, v):
        room = torch.empty(t.numel() + 4, dtype=t.dtype, device=DEV)[4:].view(t.shape)
        room.copy_(t)
        moved.append(room)
    got = ops.multimap_attention(q, *moved, AttnMeta(positions=None, slots=None, block_tables=bt, seq_lens=lens, decode=True), *args, **kw)
    want = ref.multimap_attention(q, k, v, bt, torch.arange(17, dtype=torch.int32, device=DEV), lens, *args, **kw)
    _close(got, want, vdim)


def test_shaped_heads_of_48(ops):
    """Capped and sloped heads whose pages are no whole number of KB take the splits."""
    q, k, v, bt, lens, args, kw = _case(4, 2, 1, 48, 48, "shaped", 16, 5, -1.0, seed=3)
    assert not ops.library.bcg_multimap_pairs(1, 48, 48, 1, 0)
    kp, vp = ops.kv_from_logical(k, v)
    got = ops.multimap_attention(q, kp, vp, AttnMeta(positions=None, slots=None, block_tables=bt, seq_lens=lens, decode=True), *args, **kw)
    want = ref.multimap_attention(q, k, v, bt, torch.arange(17, dtype=torch.int32, device=DEV), lens, *args, **kw)
    _close(got, want, 48)
