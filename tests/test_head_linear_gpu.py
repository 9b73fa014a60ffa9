"""The latent mixers' per-head products (csrc/kernels/seqmix_heads.hip) with the turned tail of the queries and the gate of the result, at the edges of
their tiles of tokens and columns, against fp32.  Bounds: one bf16 rounding (2^-8 of the value) beside 2^-7 where the gate rounds again, and fp32 sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _ops():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    from byzantine_consensus_llm_agents_amd.ops import reference as ref
    return get_ops("hip"), ref


def _data(T, H, K, N, tail, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, H, K + tail, generator=g).bfloat16()
    w = (torch.randn(H, K, N, generator=g) * K ** -0.5).bfloat16()
    return x, w, g


def _exact(x, w):
    return torch.bmm(x.float().transpose(0, 1), w.float()).transpose(0, 1).contiguous()


@pytest.mark.parametrize("T,H,K,N", [(1, 3, 32, 16), (63, 2, 64, 48), (64, 5, 128, 128), (65, 16, 256, 144), (300, 40, 128, 80), (5000, 30, 128, 128)])
def test_product_and_tail(T, H, K, N):
    ops, ref = _ops()
    for tail, half, pairs in ((64, 32, False), (64, 32, True), (24, 8, False), (8, 3, False)):
        x, w, g = _data(T, H, K, N, tail, T + tail)
        pos, freq = torch.randint(0, 9000, (T,), generator=g).int(), torch.rand(half, generator=g)
        dst = torch.full((T, H, N + tail), 7.0).bfloat16().to(DEV)
        got = ops.head_linear_turned(x.to(DEV), K, w.to(DEV), dst, pos.to(DEV), freq.to(DEV), 1.1, pairs).cpu()
        torch.testing.assert_close(got[:, :, :N].float(), _exact(x[:, :, :K], w), rtol=2 ** -8, atol=1e-5)
        want = ref.rope_tail(x, K, torch.zeros(T, H, N + tail).bfloat16(), N, pos, freq, 1.1, pairs)[:, :, N:]
        # (angles of up to 9000 in fp32: 2^-11 of a turn apart at worst)
        torch.testing.assert_close(got[:, :, N:].float(), want.float(), rtol=2 ** -7, atol=1e-2)


@pytest.mark.parametrize("T,H,K,N,group", [(1, 2, 32, 16, 1), (65, 3, 128, 48, 48), (129, 16, 128, 128, 1), (700, 24, 64, 96, 8), (2000, 32, 256, 64, 64)])
def test_product_and_gate(T, H, K, N, group):
    ops, ref = _ops()
    x, w, g = _data(T, H, K, N, 0, T)
    y = torch.randn(T, H * N // group + 24, generator=g).bfloat16()
    gate = y[:, 8:8 + H * N // group]
    got = ops.head_linear_gated(x.to(DEV), w.to(DEV), y.to(DEV)[:, 8:8 + H * N // group]).cpu()
    want = _exact(x, w).view(T, H * N) * torch.sigmoid(gate.float()).repeat_interleave(group, 1)
    torch.testing.assert_close(got.float(), want, rtol=2 ** -7, atol=1e-5)
    plain = ops.head_linear(x.to(DEV), w.to(DEV)).cpu()
    torch.testing.assert_close(plain.float(), _exact(x, w), rtol=2 ** -8, atol=1e-5)


# other routes keep the answers: an input width that the kernel has not, odd columns, rows off 16 bytes, fp32
@pytest.mark.parametrize("K,N,dtype,off", [(48, 32, torch.bfloat16, 0), (64, 24, torch.bfloat16, 0), (64, 32, torch.bfloat16, 1), (64, 32, torch.float32, 0)])
def test_other_operands(K, N, dtype, off):
    ops, ref = _ops()
    g = torch.Generator().manual_seed(K)
    T, H = 21, 4
    flat = torch.randn(T * H * K + off, generator=g).to(dtype).to(DEV)
    x = flat[off:].view(T, H, K)
    w = (torch.randn(H, K, N, generator=g) * K ** -0.5).to(dtype).to(DEV)
    gate = torch.randn(T, H * N, generator=g).to(dtype).to(DEV)
    want = _exact(x.cpu(), w.cpu())
    tol = dict(rtol=2 ** -7, atol=2e-2) if dtype == torch.bfloat16 else dict(rtol=1e-4, atol=1e-4)
    torch.testing.assert_close(ops.head_linear(x, w).float().cpu(), want, **tol)
    torch.testing.assert_close(ops.head_linear_gated(x, w, gate).float().cpu(), want.view(T, H * N) * torch.sigmoid(gate.float().cpu()), **tol)


def test_more_heads_than_the_grid_holds():
    ops, _ = _ops()
    x, w, _ = _data(2, 1 << 15, 32, 16, 0, 5)
    torch.testing.assert_close(ops.head_linear(x.to(DEV), w.to(DEV)).float().cpu(), _exact(x, w), rtol=2 ** -8, atol=1e-5)
