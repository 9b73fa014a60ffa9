"""The order of a decode step's rows (decode_order_kernel) against a sort, and the attention under it.  GPU only."""
import pytest
import torch

from test_decode_fused_gpu import _case, ops  # noqa: F401
from test_decode_pairs_gpu import LENS, _pairs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 2, 63, 64, 65, 255, 448, 2048])
@pytest.mark.parametrize("most", [1, 7, 5000])
def test_order(ops, B, most):
    lens = torch.randint(0, most, (B,), device="cuda", dtype=torch.int32)
    assert torch.equal(ops.decode_order(lens).long(), torch.argsort(lens, descending=True, stable=True))


@pytest.mark.parametrize("n_q,n_kv,hd,norm,parts,times", [(32, 8, 128, True, 1, 7), (14, 2, 64, False, 1, 1), (16, 1, 128, False, 2, 1)])
def test_pairs_in_any_order_are_the_same(ops, n_q, n_kv, hd, norm, parts, times):
    c, k, v, table, lens = _case(LENS[:-1] * times + [0], n_q, n_kv, hd, norm, seed=n_q + hd)
    (k0, v0), (k1, v1) = (k.clone(), v.clone()), (k.clone(), v.clone())
    want = _pairs(ops, c, k0, v0, table, lens, parts)
    got = ops.decode_attention_pairs(c["qkv"], c["positions"], c["slots"], n_q, n_kv, hd, c["q_norm"], c["k_norm"], c["eps"], c["cos_sin"], k1, v1, 1,
                                     table, lens, hd ** -0.5, None, parts, ops.decode_order(lens))
    assert torch.equal(got, want) and torch.equal(k1, k0) and torch.equal(v1, v0)
