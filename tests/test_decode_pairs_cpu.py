"""Which decode steps take a workgroup per (row, kv head) pair, and where a long row is cut.  No GPU."""
from types import SimpleNamespace

import pytest
import torch

from byzantine_consensus_llm_agents_amd.models.transformer import AttnMeta, DecoderModel
from byzantine_consensus_llm_agents_amd.ops.hip import part_rule


def test_parts():
    """(parts, one, each, ways, extra): heads of 128 have chunks of 16 KB, of 64 of 8 KB."""
    assert part_rule(80, 128 * 128, 28) == (1, 28, 8, 256, 0) and part_rule(80, 128 * 128, 29) == (4, 28, 8, 256, 240)
    assert part_rule(2, 128 * 64, 57) == (4, 56, 16, 256, 6) and part_rule(2, 128 * 64, 512) == (16, 56, 16, 256, 30)
    assert part_rule(136, 128 * 128, 128) == (1, 128, 8, 256, 0) and part_rule(136, 128 * 128, 512) == (16, 128, 8, 256, 256)
    assert part_rule(320, 128 * 128, 256) == (16, 28, 8, 1024, 1024) and part_rule(360, 128 * 128, 256)[3] == 256
    assert part_rule(16384, 128 * 128, 512) == (16, 128, 8, 256, 256) and part_rule(1, 1 << 20, 1) == (1, 0, 1, 256, 0)


@pytest.mark.parametrize("change,paired", [({}, True), ({"hd": 64}, True), ({"hd": 96}, False), ({"cascade": object()}, False), ({"decode": False}, False),
                                           ({"kv": torch.float8_e4m3fn}, False), ({"block": 32}, False), ({"strided": True}, False),
                                           ({"offset": 4}, False), ({"offset": 8}, True),
                                           ({"layer": {"qkv_s": None}}, False), ({"width": 0}, False)])   # (fp8 projections; no room for a token)
def test_route(change, paired):
    c = dict(dict(cascade=None, decode=True, rows=60, kv=torch.bfloat16, hd=128, block=16, strided=False, offset=0, layer={}, width=40), **change)
    calls = []
    ops = SimpleNamespace()
    for name in ("decode_attention_pairs", "qk_norm_rope_kv_write", "paged_attention_decode", "paged_attention_prefill"):
        setattr(ops, name, lambda *a, _n=name, **kw: calls.append(_n))
    m = object.__new__(DecoderModel)
    m.ops, m.cfg, m.hd, m.n_q, m.n_kv, m.scale, m.cos_sin = ops, SimpleNamespace(rms_eps=1e-6), c["hd"], 4, 2, 0.125, None
    i32 = torch.zeros(c["rows"], dtype=torch.int32)
    meta = AttnMeta(positions=i32, slots=i32, block_tables=torch.zeros(c["rows"], c["width"], dtype=torch.int32), seq_lens=i32, decode=c["decode"], cascade=c["cascade"])
    n = 2 * 2 * c["block"] * c["hd"]
    cache = torch.zeros(n + 8).to(c["kv"])[c["offset"]:c["offset"] + n].view(1, 2, 2, c["block"], c["hd"])
    qkv = torch.zeros(c["rows"], 8 * c["hd"], dtype=torch.bfloat16)
    m._attention(0, c["layer"], qkv.repeat(2, 1)[::2] if c["strided"] else qkv, meta, cache, cache.transpose(3, 4))
    assert calls == (["decode_attention_pairs"] if paired else
                     ["qk_norm_rope_kv_write", "paged_attention_decode" if c["decode"] else "paged_attention_prefill"])


@pytest.mark.parametrize("change,ordered", [({}, True), ({"layers": 7}, False), ({"rows": 256}, False), ({"quant": True}, False), ({"cascade": object()}, False),
                                            ({"offset": 4}, False), ({"hd": 96}, False)])
def test_order_only_for_pairs(change, ordered):
    """The launch that orders the rows comes only where the layers' attention goes by pairs."""
    c = dict(dict(layers=8, rows=257, quant=False, cascade=None, offset=0, hd=128), **change)
    calls = []
    m = object.__new__(DecoderModel)
    m.ops = SimpleNamespace(decode_attention_pairs=None, decode_order=lambda lens: calls.append(lens) or lens)
    m.hd, m.n_kv, m.layers = c["hd"], 2, [{"qkv_s": None} if c["quant"] else {}] * c["layers"]
    lens = torch.zeros(c["rows"], dtype=torch.int32)
    meta = AttnMeta(positions=lens, slots=lens, block_tables=torch.zeros(c["rows"], 4, dtype=torch.int32), seq_lens=lens, decode=True, cascade=c["cascade"])
    n = 2 * 2 * 16 * c["hd"]
    cache = torch.zeros(n + 8).to(torch.bfloat16)[c["offset"]:c["offset"] + n].view(1, 2, 2, 16, c["hd"])
    assert (m._decode_order(meta, cache, cache.transpose(3, 4)) is not None) == ordered == bool(calls)
