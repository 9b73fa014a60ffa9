"""Projections whose operands carry more than values keep the library path: shapes that the few-row kernel takes, that are
split into runs of rows and that the 256 x 256 kernel takes.  GPU only.  Bound: one bf16 rounding of an fp32 sum, 2^-8 in the
2-norm (gradients of a sum over rows: 2^-7)."""
import pytest
import torch
from torch.autograd import forward_ad

pytestmark = pytest.mark.gpu
SHAPES = [(3, 36, 128), (4449, 4096, 8192), (8183, 11264, 256)]


@pytest.fixture(scope="module")
def ops():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    return get_ops("hip")


def _data(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    return (torch.randn(M, K, device="cuda", generator=g).bfloat16(), (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16(),
            torch.randn(N, device="cuda", generator=g).bfloat16(), torch.randn(M, N, device="cuda", generator=g).bfloat16())


def _off(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_gradients_of_bias_and_residual(ops, M, N, K):
    x, w, b, r = _data(M, N, K)
    y = x.float() @ w.float().t()
    b.requires_grad_()
    out = ops.linear(x, w, b)
    assert _off(out, y + b.float()) < 2 ** -8
    out.float().sum().backward()
    assert _off(b.grad, torch.full_like(y[0], M)) < 2 ** -7
    with torch.no_grad():
        assert not ops.linear(x, w, b).requires_grad
    leaf = r.clone().requires_grad_()
    out = ops.linear_residual(x, w, leaf * 1)
    assert _off(out, y + r.float()) < 2 ** -8
    out.float().sum().backward()
    assert torch.equal(leaf.grad, torch.ones_like(leaf))


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_forward_mode(ops, M, N, K):
    x, w, b, r = _data(M, N, K)
    t = torch.ones_like(x)
    with forward_ad.dual_level():
        out = forward_ad.unpack_dual(ops.linear(forward_ad.make_dual(x, t), w))
        assert _off(out.primal, x.float() @ w.float().t()) < 2 ** -8 and _off(out.tangent, t.float() @ w.float().t()) < 2 ** -8
        out = forward_ad.unpack_dual(ops.linear(x, w, forward_ad.make_dual(b, b)))
        assert _off(out.tangent, b.expand(M, N)) < 2 ** -8


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_two_devices(ops, M, N, K):
    """One operand in host memory: refused as the library refuses it."""
    x, w, b, r = _data(M, N, K)
    for call in (lambda: ops.linear(x, w.cpu()), lambda: ops.linear(x, w, b.cpu()), lambda: ops.linear_residual(x, w, r.cpu()),
                 lambda: ops.norm_linear(x, torch.ones(K, device="cuda").bfloat16(), 1e-6, w.cpu())):
        with pytest.raises(RuntimeError):
            call()


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_autocast_and_vmap(ops, M, N, K):
    x, w, b, _ = _data(M, N, K)
    with torch.autocast("cuda", dtype=torch.float16):
        assert ops.linear(x, w, b).dtype == torch.float16
    y = torch.vmap(lambda t: ops.linear(t, w, b))(x[None])
    assert _off(y[0], x.float() @ w.float().t() + b.float()) < 2 ** -8
