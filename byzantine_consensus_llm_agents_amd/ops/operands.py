"""Which operands a kernel may take that reads and writes memory behind torch's back: where a call has a library path, that
path keeps whatever torch is asked to follow."""

import torch
from torch.autograd import forward_ad


def bare(t) -> bool:
    """Nothing is asked of the tensor but its values: no gradient and no forward-mode tangent (None: no operand)."""
    if t is None:
        return True
    if t.requires_grad and torch.is_grad_enabled():
        return False
    return forward_ad._current_level < 0 or forward_ad.unpack_dual(t).tangent is None
