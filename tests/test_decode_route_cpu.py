"""Which decode steps take the rotary embedding inside the attention launch (`DecoderModel._attention`, `decode_fused_pays`).  No GPU."""
from types import SimpleNamespace

import pytest
import torch

from byzantine_consensus_llm_agents_amd.models.transformer import AttnMeta, DecoderModel
from byzantine_consensus_llm_agents_amd.ops.hip import decode_fused_pays


def test_rule():
    assert decode_fused_pays(4, 2, 64) and decode_fused_pays(1, 16, 64)      # few heads of K and V: whatever the contexts are
    assert decode_fused_pays(96, 2, 3) and not decode_fused_pays(97, 2, 3)   # 576 parts
    assert not decode_fused_pays(100, 16, 1) and not decode_fused_pays(129, 1, 1) and not decode_fused_pays(17, 1, 64)


@pytest.mark.parametrize("change,fused", [({}, True), ({"cascade": object()}, False), ({"decode": False}, False), ({"rows": 97}, False),
                                          ({"kv": torch.float8_e4m3fn}, False), ({"hd": 128}, False), ({"block": 32}, False),
                                          ({"width": 200}, False), ({"width": 200, "rows": 8}, True), ({"strided": True}, False)])
def test_route(change, fused):
    c = dict(dict(cascade=None, decode=True, rows=60, kv=torch.bfloat16, hd=64, block=16, width=40, strided=False), **change)
    calls = []
    ops = SimpleNamespace(decode_fused_pays=lambda B, n_kv, tokens: decode_fused_pays(B, n_kv, -(-tokens // 256)))
    for name in ("decode_attention", "qk_norm_rope_kv_write", "paged_attention_decode", "paged_attention_prefill"):
        setattr(ops, name, lambda *a, _n=name, **kw: calls.append(_n))
    m = object.__new__(DecoderModel)
    m.ops, m.cfg, m.hd, m.n_q, m.n_kv, m.scale, m.cos_sin = ops, SimpleNamespace(rms_eps=1e-6), c["hd"], 4, 2, 0.125, None
    i32 = torch.zeros(c["rows"], dtype=torch.int32)
    meta = AttnMeta(positions=i32, slots=i32, block_tables=torch.zeros(c["rows"], c["width"], dtype=torch.int32), seq_lens=i32, decode=c["decode"],
                    cascade=c["cascade"])
    cache = torch.zeros(1, 2, 2, c["block"], c["hd"]).to(c["kv"])
    qkv = torch.zeros(c["rows"], 8 * c["hd"], dtype=torch.bfloat16)
    m._attention(0, {}, qkv.repeat(2, 1)[::2] if c["strided"] else qkv, meta, cache, cache.transpose(3, 4))
    assert calls == (["decode_attention"] if fused else ["qk_norm_rope_kv_write", "paged_attention_decode" if c["decode"] else "paged_attention_prefill"])
