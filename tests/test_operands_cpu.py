"""Which operands the kernels without a graph behind them take (ops/operands.py), without a GPU."""
import torch
from torch.autograd import forward_ad

from byzantine_consensus_llm_agents_amd.ops.operands import bare


def test_gradients_and_tangents():
    x, p = torch.ones(2, 3), torch.nn.Parameter(torch.ones(2, 3))
    assert bare(None) and bare(x) and not bare(p) and not bare(p * 2)
    with torch.no_grad():
        assert bare(p)
    with torch.inference_mode():
        assert bare(p)
    with forward_ad.dual_level():
        assert bare(x) and not bare(forward_ad.make_dual(x, torch.ones_like(x)))
    assert bare(x)
