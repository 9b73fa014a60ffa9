"""bf16 values that a kernel passes on without arithmetic keep all their bits: subnormal numbers, which the build flushes where it computes, and NaN
payloads among them.  GPU only."""
import pytest
import torch

from test_row_kernels_gpu import ops  # noqa: F401

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _bits(*shape):
    """Every bf16 pattern in turn, subnormal numbers at every third place."""
    n = torch.Size(shape).numel()
    a = torch.arange(n, device=DEV) * 40503 % 65536
    a = torch.where(torch.arange(n, device=DEV) % 3 == 0, a & 0x807f, a)
    return torch.where(a >= 32768, a - 65536, a).to(torch.int16).view(*shape)


def _same(x, bits):
    assert torch.equal(x.contiguous().view(torch.int16), bits.contiguous())


@pytest.mark.parametrize("T,H", [(5, 64), (5, 4096), (300, 2048), (300, 5120), (7, 8192)])
def test_rows_into_the_stream(ops, T, H):
    rows = _bits(T, H)
    x, w = rows.view(torch.bfloat16), torch.ones(H, device=DEV, dtype=torch.bfloat16)
    tokens = torch.arange(T, device=DEV, dtype=torch.int32).flip(0)
    _same(ops.add_rmsnorm(x, None, w, 1e-5)[1], rows)
    _same(ops.embed_rmsnorm(tokens, x, w, 1e-5)[1], rows.flip(0))
    _same(ops.add_rmsnorm_fp8(x, None, w, 1e-5)[2], rows)
    _same(ops.embed_rmsnorm_fp8(tokens, x, w, 1e-5)[2], rows.flip(0))


@pytest.mark.parametrize("hd", [64, 96, 128])
@pytest.mark.parametrize("T,contiguous", [(9, False), (40, True)])
def test_decoder_values(ops, hd, T, contiguous):
    n_q, n_kv, NB = 4, 2, 5
    qkv = _bits(T, (n_q + 2 * n_kv) * hd)
    k, v = torch.zeros(1, NB, n_kv, 16, hd, device=DEV, dtype=torch.bfloat16), torch.zeros(1, NB, n_kv, hd, 16, device=DEV, dtype=torch.bfloat16)
    slots = torch.arange(11, 11 + T, device=DEV, dtype=torch.int32)
    cos_sin = torch.rand(128, hd, device=DEV)
    ops.qk_norm_rope_kv_write(qkv.view(torch.bfloat16), slots, slots, n_q, n_kv, hd, None, None, 1e-6, cos_sin, k, v, 0, contiguous=contiguous)
    _same(v[0].permute(0, 3, 1, 2).reshape(NB * 16, n_kv * hd)[11:11 + T], qkv[:, (n_q + n_kv) * hd:])


@pytest.mark.parametrize("dim,rot", [(64, 32), (20, 12), (32, 0)])   # (four features an access, the halves not in fours)
@pytest.mark.parametrize("T", [9, 1100])
def test_unturned_features(ops, dim, rot, T):
    n_q, n_kv, maps, vdim, NB = 3, 2, 2, 32, 80
    qw, kw = n_q * maps * dim, n_kv * maps * dim
    x = _bits(T, qw + kw + n_kv * vdim)
    k, v = torch.zeros(NB, n_kv, 16, maps * dim, device=DEV, dtype=torch.bfloat16), torch.zeros(NB, n_kv, vdim, 16, device=DEV, dtype=torch.bfloat16)
    slots = torch.arange(11, 11 + T, device=DEV, dtype=torch.int32)
    inv = torch.rand(rot // 2, device=DEV)
    q = ops.rope_multi_kv_write(x.view(torch.bfloat16), slots, slots, n_q, n_kv, maps, dim, vdim, inv, k, v)
    kl, vl = ops.kv_to_logical(k, v)
    kl, vl = (t.reshape(NB * 16, -1)[11:11 + T] for t in (kl.permute(0, 2, 1, 3), vl.permute(0, 3, 1, 2)))
    _same(q.view(T, n_q * maps, dim)[:, :, rot:], x[:, :qw].view(T, n_q * maps, dim)[:, :, rot:])
    _same(kl.view(T, n_kv * maps, dim)[:, :, rot:], x[:, qw:qw + kw].view(T, n_kv * maps, dim)[:, :, rot:])
    _same(vl, x[:, qw + kw:])


def test_latent_key_part(ops):
    T, R, RD, half, NB = 23, 64, 32, 8, 4
    y = _bits(T, R + RD)
    k, v = torch.zeros(NB, 1, 16, R + RD, device=DEV, dtype=torch.bfloat16), torch.zeros(NB, 1, R, 16, device=DEV, dtype=torch.bfloat16)
    slots = torch.arange(11, 11 + T, device=DEV, dtype=torch.int32)
    ops.latent_kv_write(y.view(torch.bfloat16), 0, R, RD, torch.ones(R, device=DEV), 1e-5, slots, slots, torch.rand(half, device=DEV), 1.1, k, v, True)
    kl, _ = ops.kv_to_logical(k, v)
    _same(kl.reshape(NB * 16, R + RD)[11:11 + T, R + 2 * half:], y[:, R + 2 * half:])


@pytest.mark.parametrize("half", [0, 8])
def test_values_beside_pairs(ops, half):
    T, H, G, dim, vdim, NB = 23, 2, 1, 32, 48, 4
    x = _bits(T, (H + G) * dim + G * vdim)
    k, v = torch.zeros(NB, G, 16, dim, device=DEV, dtype=torch.bfloat16), torch.zeros(NB, G, vdim, 16, device=DEV, dtype=torch.bfloat16)
    slots = torch.arange(11, 11 + T, device=DEV, dtype=torch.int32)
    ops.rope_pairs_kv_write(x.view(torch.bfloat16), slots, slots, H, G, dim, vdim, None, None, 1e-5, torch.rand(half, device=DEV), None, k, v)
    _, vl = ops.kv_to_logical(k, v)
    _same(vl.permute(0, 3, 1, 2).reshape(NB * 16, G * vdim)[11:11 + T], x[:, (H + G) * dim:])
