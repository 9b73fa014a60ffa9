"""Prefill attention with the pages staged through LDS, at the edges of its 32-key chunks, 16-row waves and 64-row tiles
and with every mask it takes, against the reference.  GPU only.  Bound: outputs are averages of unit normals under
weights rounded to bf16 once (2^-9 each, so at most 2^-9 of the largest |v| ~ 4) and rounded to bf16 once: 2e-2."""
import pytest
import torch

from byzantine_consensus_llm_agents_amd.ops import reference as ref
from test_seqmix_kernels_gpu import _paged

pytestmark = pytest.mark.gpu

SEQ = [1000, 64, 65, 31, 33, 16, 17, 2, 130, 48]
NEW = [129, 64, 65, 31, 2, 16, 17, 2, 63, 47]


@pytest.fixture(scope="module")
def ops():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    return get_ops("hip")


@pytest.mark.parametrize("maps,dim,vdim", [(1, 32, 32), (1, 48, 48), (1, 64, 128), (1, 128, 128), (1, 192, 128), (1, 256, 256),
                                           (2, 64, 128), (2, 48, 96), (2, 32, 32)])
@pytest.mark.parametrize("H,G", [(4, 2), (3, 1)])
@pytest.mark.parametrize("kind", ["plain", "window", "chunk", "sink", "shaped", "keep"])
def test_staged_prefill(ops, maps, dim, vdim, H, G, kind):
    if maps == 2 and kind != "plain":
        pytest.skip("masks and sinks: one-map heads")
    k, v, meta, T = _paged(SEQ, NEW, 16, G, maps * dim, vdim, torch.bfloat16, seed=dim)
    dev = k.device
    q = torch.randn(T, H, maps * dim, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(dev)
    kw = dict(plain={}, window=dict(window=37), chunk=dict(chunk=50), sink=dict(sink=torch.randn(H, device=dev), window=100),
              shaped=dict(softcap=3.0, slopes=torch.rand(H, device=dev) * 0.1), keep=dict(window=40, keep=5))[kind]
    args = (dim ** -0.5, maps, 0.35, -1.0, 1.0, vdim)
    got = ops.multimap_attention(q, *ops.kv_from_logical(k, v), meta, *args, **kw)
    want = ref.multimap_attention(q.float(), k.float(), v.float(), meta.block_tables, meta.q_start, meta.seq_lens, *args, **kw)
    torch.testing.assert_close(got.float(), want.float().reshape(got.shape), rtol=2e-2, atol=2e-2)


def test_entries_without_rows(ops):
    """A tile list padded with entries that hold no row, their sequence and row outside the batch: nothing of them is read."""
    k, v, meta, T = _paged(SEQ, NEW, 16, 2, 64, 128, torch.bfloat16, seed=3)
    q = torch.randn(T, 4, 64, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(k.device)
    args = (0.125, 1, 0.0, -1.0, 1.0, 128)
    want = ops.multimap_attention(q, *ops.kv_from_logical(k, v), meta, *args)
    pad = torch.tensor([[-1, T, T], [len(SEQ), 0, 0], [0, 5, 5]], dtype=torch.int32, device=k.device)
    meta.tiles = torch.cat([pad, meta.tiles, pad])
    assert torch.equal(ops.multimap_attention(q, *ops.kv_from_logical(k, v), meta, *args), want)


def test_caches_off_16_bytes(ops):
    """Caches 8 bytes past a 16-byte boundary: the same kernel, the same bits."""
    k, v, meta, T = _paged(SEQ, NEW, 16, 2, 64, 128, torch.bfloat16, seed=3)
    q = torch.randn(T, 4, 64, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(k.device)
    args = (0.125, 1, 0.0, -1.0, 1.0, 128)
    kl, vl = ops.kv_from_logical(k, v)
    off = [torch.cat([x.new_zeros(4), x.flatten()])[4:].view(x.shape) for x in (kl, vl)]
    assert all(x.data_ptr() % 16 == 8 for x in off)
    assert torch.equal(ops.multimap_attention(q, *off, meta, *args), ops.multimap_attention(q, kl, vl, meta, *args))


def test_more_workgroups_than_one_dimension_holds(ops):
    """2^24 tiles x heads of 256 threads do not fit a one-dimensional launch: such calls keep the general instances."""
    H = 17
    k, v, meta, T = _paged([16], [16], 16, 1, 32, 32, torch.bfloat16, seed=3)
    q = torch.randn(T, H, 32, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(k.device)
    args = (32 ** -0.5, 1, 0.0, -1.0, 1.0, 32)
    want = ops.multimap_attention(q, *ops.kv_from_logical(k, v), meta, *args)
    meta.tiles = torch.cat([meta.tiles, torch.tensor([[0, 0, 0]], dtype=torch.int32, device=k.device).expand((1 << 24) // H, 3)]).contiguous()
    got = ops.multimap_attention(q, *ops.kv_from_logical(k, v), meta, *args)
    torch.testing.assert_close(got, want, rtol=2e-2, atol=2e-2)
