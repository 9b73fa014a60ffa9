"""Row kernels at the edges of their variants (rows in registers, several columns per access, several tokens per
workgroup) against the reference ops.  GPU only.  Bounds: fp32 sums in another order 1e-5, one bf16 rounding 2^-8; whole
fp8 rows match up to single values that round the other way (an exp of the last bit)."""
import types

import pytest
import torch

from byzantine_consensus_llm_agents_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    return get_ops("hip")


def _tol(dtype):
    return dict(rtol=2 ** -7, atol=1e-2) if dtype == torch.bfloat16 else dict(rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W", [4, 1020, 2048, 2052, 4100, 8192, 8196, 2050])
def test_embed_and_residual_rows(ops, dtype, W):
    g = torch.Generator(device="cuda").manual_seed(W)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    T = 5
    table, w, add = r(50, W).to(dtype), r(W) * 0.1, r(W)
    tokens = torch.randint(0, 50, (T,), device="cuda", generator=g, dtype=torch.int32)
    for a in (None, add):
        for x, y in zip(ops.embed_scale_rmsnorm(tokens, table, 0.7, w, 1e-5, 1.0, dtype, a),
                        ref.embed_scale_rmsnorm(tokens, table, 0.7, w, 1e-5, 1.0, dtype, a)):
            torch.testing.assert_close(x, y, **_tol(dtype))
    x, p, f, gate = r(T, W), [r(T, W).to(dtype) for _ in range(3)], r(T, W), r(T)
    for parts, gt, gd in (([p[0]], None, None), ([p[0], f], gate, p[2]), ([p[0], p[1]], None, None)):
        xa, xb = x.clone(), x.clone()
        torch.testing.assert_close(ops.residual_add_rmsnorm32(xa, parts, w, 1e-5, 1.0, dtype, gt, gd),
                                   ref.residual_add_rmsnorm32(xb, parts, w, 1e-5, 1.0, dtype, gt, gd), **_tol(dtype))
        torch.testing.assert_close(xa, xb, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["gelu_tanh", "relu2", "silu"])
@pytest.mark.parametrize("rows,n,stride,off", [(1, 8, 8, 0), (3, 2056, 4096, 8), (70000, 8, 24, 16), (5, 100, 104, 0), (5, 96, 104, 4)])
def test_activation_columns(ops, dtype, kind, rows, n, stride, off):
    z = torch.randn(rows, stride, device="cuda").to(dtype) * 4
    z[0, off], z[-1, off + 1] = 200.0, -200.0
    view = z[:, off:off + n]
    torch.testing.assert_close(ops.act_fn(view, kind), ref.act_fn(view, kind), rtol=2 ** -7 if dtype == torch.bfloat16 else 1e-5,
                               atol=1e-6 if dtype == torch.float32 else 1e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n_q,n_kv,maps,dim,vdim,rot", [(4, 2, 2, 64, 128, 64), (3, 1, 1, 20, 12, 16), (2, 2, 2, 32, 8, 0), (2, 1, 1, 24, 32, 12)])
@pytest.mark.parametrize("T", [1, 7, 1023, 1024, 1031])
def test_rope_tokens_of_a_group(ops, dtype, n_q, n_kv, maps, dim, vdim, rot, T):
    """Runs of slots that start inside a 4-key group, end in one, jump, and a token without a slot in the pool."""
    BS, NB = 16, 1 + (T + 40) // 16
    half = rot // 2
    inv = (10000.0 ** (-torch.arange(half, device="cuda") / max(half, 1))).float()
    width = n_q * maps * dim + n_kv * maps * dim + n_kv * vdim
    x = torch.randn(T, width + 8, device="cuda").to(dtype)
    slots = torch.arange(3, 3 + T, device="cuda", dtype=torch.int32)
    if T > 16:
        slots[T // 2:] += 7
    pos = slots * 3
    shape_k, shape_v = (NB, n_kv, BS, maps * dim), (NB, n_kv, vdim, BS)
    k, v = torch.zeros(shape_k, device="cuda", dtype=dtype), torch.zeros(shape_v, device="cuda", dtype=dtype)
    q = ops.rope_multi_kv_write(x, pos, slots, n_q, n_kv, maps, dim, vdim, inv, k, v)
    kr, vr = torch.zeros(shape_k, device="cuda", dtype=dtype), torch.zeros(shape_v, device="cuda", dtype=dtype)
    qr = ref.rope_multi_kv_write(x, pos, slots, n_q, n_kv, maps, dim, vdim, inv, kr, vr)
    # fragment-major slabs back to the reference's layout
    k = k.view(NB, n_kv, maps * dim // 4, BS, 4).permute(0, 1, 3, 2, 4).reshape(shape_k)
    v = v.view(NB, n_kv, BS // 4, vdim, 4).permute(0, 1, 3, 2, 4).reshape(shape_v)
    tol = dict(rtol=2 ** -7, atol=1e-2) if dtype == torch.bfloat16 else dict(rtol=1e-4, atol=1e-4)
    torch.testing.assert_close(q.reshape(qr.shape), qr, **tol)
    torch.testing.assert_close(k, kr, **tol)
    assert torch.equal(v, vr)


@pytest.mark.parametrize("splits,vdim,maps", [(1, 128, 2), (9, 128, 1), (9, 33, 1), (70, 48, 1)])
def test_merge_of_splits(ops, splits, vdim, maps):
    """Contexts of up to more than 64 splits, odd value widths, contexts of one key beside long ones."""
    n, G, H, dim, BS = 3, 1, 2, 16, 16
    ctx = [1, splits * 128 - 5, (splits - 1) * 128 + 1]
    nblk = -(-max(ctx) // BS)
    tables = torch.arange(1, 1 + n * nblk, device="cuda", dtype=torch.int32).view(n, nblk)
    g = torch.Generator(device="cuda").manual_seed(splits)
    dt = torch.float32
    k = torch.randn(n * nblk + 1, G, BS, maps * dim, device="cuda", generator=g)
    v = torch.randn(n * nblk + 1, G, vdim, BS, device="cuda", generator=g)
    q = torch.randn(n, H, maps * dim, device="cuda", generator=g)
    meta = types.SimpleNamespace(block_tables=tables, seq_lens=torch.tensor(ctx, device="cuda", dtype=torch.int32), decode=True,
                                 attn_seq_lens=None, q_start=None, tiles=None, single=None, tile_rows=64, positions=None)
    out = ops.multimap_attention(q, k, v, meta, 0.3, maps, 0.4 if maps == 2 else 0.0, -1.0, 1.0, vdim)
    kl = k.view(-1, G, maps * dim // 4, BS, 4).permute(0, 1, 3, 2, 4).reshape(k.shape)
    vl = v.view(-1, G, BS // 4, vdim, 4).permute(0, 1, 3, 2, 4).reshape(v.shape)
    for b, c in enumerate(ctx):
        kk = kl[tables[b].long()].transpose(1, 2).reshape(-1, G, maps, dim)[:c].double()
        vv = vl[tables[b].long()].permute(0, 3, 1, 2).reshape(-1, G, vdim)[:c, 0].double()
        for h in range(H):
            o = 0.0
            for m in range(maps):
                p = torch.softmax(kk[:, 0, m] @ q[b, h].double().view(maps, dim)[m] * 0.3, 0)
                o = o + (1.0 if m == 0 else -0.4) * (p @ vv)
            torch.testing.assert_close(out.view(n, H, vdim)[b, h].double(), o, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("T", [1, 256, 257])
@pytest.mark.parametrize("I", [16, 8192, 8208, 16384, 16400])
def test_fp8_rows(ops, T, I):
    gu = torch.randn(T, 2 * I, device="cuda").bfloat16()
    q, s = ops.silu_mul_fp8(gu)
    qr, sr = ref.silu_mul_fp8(gu)
    torch.testing.assert_close(s, sr, rtol=2 ** -7, atol=0)
    back, want = q.float() * s[:, None], qr.float() * sr[:, None]
    assert ((back - want).norm() / want.norm()).item() < 0.02
    if I <= 8192:
        x, res = (torch.randn(T, I, device="cuda").bfloat16() for _ in range(2))
        w = torch.randn(I, device="cuda").bfloat16()
        a, b = ops.add_rmsnorm_fp8(x, res.clone(), w, 1e-6), ref.add_rmsnorm_fp8(x, res.clone(), w, 1e-6)
        assert torch.equal(a[2], b[2])
        torch.testing.assert_close(a[1], b[1], rtol=2 ** -7, atol=0)
        back, want = a[0].float() * a[1][:, None], b[0].float() * b[1][:, None]
        assert ((back - want).norm() / want.norm()).item() < 0.02


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,vdim", [(3, 4), (2, 64), (5, 68), (4, 128), (3, 132), (2, 256), (2, 260), (1, 1024), (1, 1028), (3, 66)])
@pytest.mark.parametrize("form", ["plain", "gated", "offset", "whole-row weight"])
def test_head_norm_rows(ops, dtype, H, vdim, form):
    g = torch.Generator(device="cuda").manual_seed(vdim)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    T = 7
    o, w = r(T, H, vdim), r(H * vdim if form == "whole-row weight" else vdim)
    gate = None if form == "plain" else r(T, H * vdim + 8).to(dtype)[:, (2 if form == "offset" else 8):][:, :H * vdim]
    for act in ("sigmoid", "silu"):
        a = (o, None if form == "plain" else w, 1e-5, gate, dtype, act)
        torch.testing.assert_close(ops.head_norm_gate(*a), ref.head_norm_gate(*a), **_tol(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,vdim,parts", [(2, 4, 2), (16, 64, 1), (17, 64, 1), (33, 64, 1), (65, 64, 1), (129, 64, 1), (4, 66, 2), (130, 64, 2)])
def test_gated_group_rows(ops, dtype, H, vdim, parts):
    g = torch.Generator(device="cuda").manual_seed(H)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    T, n = 5, H * vdim
    for off in (0, 2):
        a = (r(T, H, vdim), r(T, n + 8).to(dtype)[:, off:off + n], r(H), r(T, n + 4).to(dtype)[:, :n], r(n), parts, 1e-5, dtype)
        torch.testing.assert_close(ops.gated_group_norm(*a), ref.gated_group_norm(*a), **_tol(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W", [4, 1020, 2052, 2050])
def test_embed_dyt_rows(ops, dtype, W):
    table, w, b = torch.randn(50, W, device="cuda").to(dtype), torch.randn(W, device="cuda"), torch.randn(W, device="cuda")
    tokens = torch.randint(0, 50, (5,), device="cuda", dtype=torch.int32)
    a = (tokens, table, 0.7, (0.8, w, b), dtype)
    for x, y in zip(ops.embed_scale_dyt(*a), ref.embed_scale_dyt(*a)):
        torch.testing.assert_close(x, y, **_tol(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps", [2, 3, 4])
def test_short_conv_blocks_of_rows(ops, dtype, taps):
    """Large steps: blocks of rows inside a segment, over a boundary, at a segment's first rows, a continued segment."""
    from test_decay_chunks_gpu import _meta
    lens, starts, C = [1001, 1, 2, 7, 1040, 9], [0, 4, 0, 3, 11, 0], 40
    meta, T = _meta(lens, starts, "cuda"), sum(lens)
    y = torch.randn(T, C + 8, device="cuda").to(dtype)
    w, b = torch.randn(C, taps, device="cuda"), torch.randn(C, device="cuda")
    sa = torch.randn(len(lens) + 2, taps - 1, C, device="cuda").to(dtype)
    sb = sa.clone()
    torch.testing.assert_close(ops.short_conv(y, C, w, meta, sa, "silu", b), ref.short_conv(y, C, w, meta, sb, "silu", b), **_tol(dtype))
    torch.testing.assert_close(sa, sb, rtol=0, atol=0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,dim", [(2, 1, 4), (6, 3, 100), (4, 2, 128), (2, 2, 132), (2, 1, 30)])
def test_delta_prepare_rows(ops, dtype, H, G, dim):
    T = 5
    r = lambda *s: torch.randn(*s, device="cuda")  # noqa: E731
    c, y, a = r(T, 2 * G * dim + 8).to(dtype), r(T, H + 3).to(dtype), r(T, H).to(dtype)
    args = (c, y, 2, a, r(H), r(H), H, G, dim)
    for x, z in zip(ops.delta_prepare(*args), ref.delta_prepare(*args)):
        torch.testing.assert_close(x, z, rtol=2e-5, atol=1e-5)
