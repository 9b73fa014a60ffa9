"""Which decode steps take a workgroup per (row, kv head) pair, and in how many parts.  No GPU."""
from types import SimpleNamespace

import pytest
import torch

from byzantine_consensus_llm_agents_amd.models.transformer import AttnMeta, DecoderModel
from byzantine_consensus_llm_agents_amd.ops.hip import decode_parts


def test_parts():
    assert decode_parts(10, 8, 128, 896) == 1 and decode_parts(10, 8, 128, 912) == 3
    assert decode_parts(1, 2, 64, 1792) == 1 and decode_parts(1, 2, 64, 1808) == 4 and decode_parts(1, 2, 64, 16384) == 16
    assert decode_parts(17, 8, 128, 16384) == 1 and decode_parts(2048, 8, 128, 8192) == 1


@pytest.mark.parametrize("change,paired", [({}, True), ({"hd": 64}, True), ({"hd": 96}, False), ({"cascade": object()}, False), ({"decode": False}, False),
                                           ({"kv": torch.float8_e4m3fn}, False), ({"block": 32}, False), ({"strided": True}, False),
                                           ({"offset": 4}, False), ({"offset": 8}, True),
                                           ({"layer": {"qkv_s": None}}, False)])   # (fp8 projections)
def test_route(change, paired):
    c = dict(dict(cascade=None, decode=True, rows=60, kv=torch.bfloat16, hd=128, block=16, strided=False, offset=0, layer={}), **change)
    calls = []
    ops = SimpleNamespace()
    for name in ("decode_attention_pairs", "qk_norm_rope_kv_write", "paged_attention_decode", "paged_attention_prefill"):
        setattr(ops, name, lambda *a, _n=name, **kw: calls.append(_n))
    m = object.__new__(DecoderModel)
    m.ops, m.cfg, m.hd, m.n_q, m.n_kv, m.scale, m.cos_sin = ops, SimpleNamespace(rms_eps=1e-6), c["hd"], 4, 2, 0.125, None
    i32 = torch.zeros(c["rows"], dtype=torch.int32)
    meta = AttnMeta(positions=i32, slots=i32, block_tables=torch.zeros(c["rows"], 40, dtype=torch.int32), seq_lens=i32, decode=c["decode"], cascade=c["cascade"])
    n = 2 * 2 * c["block"] * c["hd"]
    cache = torch.zeros(n + 8).to(c["kv"])[c["offset"]:c["offset"] + n].view(1, 2, 2, c["block"], c["hd"])
    qkv = torch.zeros(c["rows"], 8 * c["hd"], dtype=torch.bfloat16)
    m._attention(0, c["layer"], qkv.repeat(2, 1)[::2] if c["strided"] else qkv, meta, cache, cache.transpose(3, 4))
    assert calls == (["decode_attention_pairs"] if paired else
                     ["qk_norm_rope_kv_write", "paged_attention_decode" if c["decode"] else "paged_attention_prefill"])
