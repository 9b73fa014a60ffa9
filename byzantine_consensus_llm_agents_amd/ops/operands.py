"""Which operands a kernel may take that reads and writes memory behind torch's back: where a call has a library path, that
path keeps whatever torch is asked to follow."""

import torch
from torch.autograd import forward_ad

PLAIN = (torch.Tensor, torch.nn.Parameter)


def watched() -> bool:
    """Somebody follows the calls themselves: a trace, a dispatch mode (fakes, proxies, counters), autocast."""
    return (torch._C._len_torch_dispatch_stack() > 0 or torch.jit.is_tracing() or torch.compiler.is_compiling()
            or torch.is_autocast_enabled("cuda"))


def bare(t) -> bool:
    """The tensor is its memory and nothing is asked of it but its values: no subclass, no wrapper of a transform (vmap,
    functional gradients), no gradient, no forward-mode tangent (None: no operand)."""
    if t is None:
        return True
    if type(t) not in PLAIN or (t.requires_grad and torch.is_grad_enabled()):
        return False
    try:
        t.data_ptr()
    except RuntimeError:   # a wrapper: no memory of its own
        return False
    return forward_ad._current_level < 0 or forward_ad.unpack_dual(t).tangent is None
