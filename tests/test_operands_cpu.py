"""Which operands the kernels without a graph behind them take (ops/operands.py), without a GPU."""
import os

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.autograd import forward_ad
from torch.fx.experimental.proxy_tensor import make_fx

from byzantine_consensus_llm_agents_amd.ops import get_ops
from byzantine_consensus_llm_agents_amd.ops.operands import bare, watched
from byzantine_consensus_llm_agents_amd.utils.build import kernels_target


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


@pytest.fixture(scope="module")
def ops():
    if not os.path.exists(kernels_target()):
        pytest.skip("kernel library not built")
    ops = get_ops("hip")
    if ops.gemm_plan.mode != "1":
        pytest.skip("BCG_HAND_GEMM")
    return ops


def _data():
    g = torch.Generator().manual_seed(1)
    return [torch.randn(*s, generator=g).bfloat16() for s in ((5, 3, 128), (36, 128), (36,), (5, 3, 36))]


def test_host_memory(ops):
    """Operands in host memory, or on two devices, never reach a kernel: the library computes them, or says no."""
    x, w, b, r = _data()
    want = torch.nn.functional.linear(x[0], w, b)
    assert torch.equal(ops.linear(x[0], w, b), want)
    assert torch.equal(ops.linear_residual(x[0], w, r[0].clone()), r[0].addmm(x[0], w.t()))
    rows, wide = x.reshape(15, 128)[:1].expand(2900, 128).contiguous(), w[:1].expand(24576, 128).contiguous()
    assert ops.gemm_plan.pieces(2900, 24576, 128, 0)[0][1] is not None     # (a shape of the 256 x 256 kernel)
    assert torch.equal(ops.linear(rows, wide), torch.nn.functional.linear(rows, wide))


def test_transforms(ops):
    """The few-row kernel's shapes under vmap, functional gradients and tangents, as the library computes them."""
    lin = torch.nn.functional.linear
    x, w, b, r = _data()
    assert torch.equal(torch.vmap(lambda t: ops.linear(t, w, b))(x), torch.vmap(lambda t: lin(t, w, b))(x))
    two = torch.stack([w, -w])
    assert torch.equal(torch.vmap(lambda t: ops.linear(x[0], t))(two), torch.vmap(lambda t: lin(x[0], t))(two))
    got, want = (torch.vmap(f)(x, r.clone()) for f in (lambda t, u: ops.linear_residual(t, w, u), lambda t, u: u.addmm_(t, w.t())))
    assert torch.equal(got, want)
    for arg in range(3):
        a = (x[0], w, b)
        got = torch.func.grad(lambda t: ops.linear(*a[:arg], t, *a[arg + 1:]).float().sum())(a[arg])
        assert torch.equal(got, torch.func.grad(lambda t: lin(*a[:arg], t, *a[arg + 1:]).float().sum())(a[arg]))
    got, want = (torch.func.jvp(lambda t: f(t, w, b), (x[0],), (x[1],)) for f in (ops.linear, lin))
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_traces_and_fakes(ops):
    x, w, b, _ = _data()
    x = x[0]
    f = lambda x, w, b: ops.linear(x, w, b)  # noqa: E731
    for trace in (make_fx(f)(x, w, b), make_fx(f, tracing_mode="fake")(x, w, b), torch.jit.trace(f, (x, w, b))):
        assert torch.equal(trace(x * 2, w, b), torch.nn.functional.linear(x * 2, w, b))
    with FakeTensorMode() as mode:
        assert watched() and ops.linear(mode.from_tensor(x), mode.from_tensor(w)).shape == (3, 36)
    assert not watched() and not bare(mode.from_tensor(x))


def test_small_steps_are_not_looked_at(ops, monkeypatch):
    """From 17 rows to LARGE_M a projection is one run whatever its operands are: no check is paid for there."""
    from byzantine_consensus_llm_agents_amd.ops import hip
    from byzantine_consensus_llm_agents_amd.ops.gemm_plan import LARGE_M
    seen = []
    monkeypatch.setattr(hip, "bare", lambda t: seen.append(t) or bare(t))
    w, b = torch.ones(36, 128).bfloat16(), torch.ones(36).bfloat16()
    for M in (17, 100, LARGE_M - 1):
        x, r = torch.ones(M, 128).bfloat16(), torch.zeros(M, 36).bfloat16()
        ops.linear(x, w, b)
        ops.linear_residual(x, w, r)
    assert not seen
