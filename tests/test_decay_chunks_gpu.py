"""The recurrence with one decay per head in chunks of 64 tokens against the token-by-token reference in float64, at the
edges of blocks, chunks and tiles and for decays from 0 to 1.  GPU only.  Bound: fp32 products and sums of at most 300 + 1
terms in another order, 1e-5 of the largest partial sum (|q|, |k| unit, |v|, |beta| of a few units)."""
import math

import pytest
import torch

from byzantine_consensus_llm_agents_amd.models.transformer import AttnMeta
from byzantine_consensus_llm_agents_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    return get_ops("hip")


def _meta(lens, starts, dev):
    i32 = torch.int32
    q = [0]
    for n in lens:
        q.append(q[-1] + n)
    t = lambda x: torch.tensor(x, dtype=i32, device=dev)  # noqa: E731
    return AttnMeta(positions=t([p for n, s in zip(lens, starts) for p in range(s, s + n)]), slots=None, block_tables=None,
                    seq_lens=t([s + n for n, s in zip(lens, starts)]), decode=False, q_start=t(q),
                    state_rows=t(list(range(len(lens), 0, -1))), token_seq=t([b for b, n in enumerate(lens) for _ in range(n)]))


def _inputs(lens, H, Gq, dim, vdim, dtype, decay, seed=0):
    g = torch.Generator().manual_seed(seed)
    T = sum(lens)
    q, k = (torch.nn.functional.normalize(torch.randn(T, Gq, dim, generator=g), dim=-1) for _ in range(2))
    v = torch.randn(T, H * vdim + 8, generator=g).to(dtype)[:, 3:3 + H * vdim]
    if decay == "fixed":
        d, beta = torch.linspace(0, 1, H), None
    else:
        d = torch.exp(-torch.exp(4 * torch.randn(T, H, 1, generator=g) - 2))   # from about 0 to about 1
        d[::37] = 0.0
        d[1::41] = 1.0
        beta = torch.rand(T, H, generator=g) * 2
    state = torch.randn(len(lens) + 2, H, dim, vdim, generator=g)
    return q, k, d, v, beta, state


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,Gq,dim,vdim", [(4, 1, 128, 64), (2, 2, 64, 80), (3, 3, 20, 18), (2, 1, 256, 33), (130, 2, 32, 64)])
@pytest.mark.parametrize("decay", ["fixed", "token"])
def test_chunks(ops, dtype, H, Gq, dim, vdim, decay):
    lens, starts = [300, 1, 16, 64, 15, 65, 17, 129], [0, 5, 3, 0, 7, 64, 0, 9]
    q, k, d, v, beta, state = _inputs(lens, H, Gq, dim, vdim, dtype, decay)
    want_state = state.double()
    want = ref.gated_state_scan(q.double(), k.double(), d.double(), v.double(), None if beta is None else beta.double(),
                                _meta(lens, starts, "cpu"), want_state, False)
    c = lambda x: None if x is None else x.to(DEV)  # noqa: E731
    got_state = c(state)
    got = ops.gated_state_scan(c(q), c(k), c(d), c(v), c(beta), _meta(lens, starts, DEV), got_state, False)
    bound = 1e-5 * (8 + 4 * math.sqrt(300))
    torch.testing.assert_close(got.cpu().double(), want.double(), rtol=0, atol=bound)
    torch.testing.assert_close(got_state.cpu().double(), want_state, rtol=0, atol=bound)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_values_out_of_range_stay_behind_their_token(ops, dtype):
    """An infinite or NaN value reaches its own and later tokens of its segment, no earlier one and no other segment."""
    lens, starts = [100, 90], [0, 0]
    q, k, d, v, beta, state = _inputs(lens, 2, 1, 64, 64, dtype, "token", 1)
    d.clamp_(min=0.5)
    clean = ops.gated_state_scan(*(x.to(DEV) for x in (q, k, d)), v.to(DEV), beta.to(DEV), _meta(lens, starts, DEV), state.to(DEV), False)
    for bad in (math.inf, math.nan):
        w = v.clone()
        w[70, 5] = bad
        got = ops.gated_state_scan(*(x.to(DEV) for x in (q, k, d)), w.to(DEV), beta.to(DEV), _meta(lens, starts, DEV), state.to(DEV), False)
        keep = torch.ones_like(got, dtype=torch.bool)
        keep[70:100, 0, 5] = False
        torch.testing.assert_close(got[keep], clean[keep], rtol=0, atol=1e-4)
        assert not torch.isfinite(got[70:100, 0, 5]).any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dim", [1, 12, 16, 33, 48, 65, 80, 96, 130, 176])
def test_what_lies_past_the_key_features(ops, dtype, dim):
    """Widths that leave whole 16-feature tiles unused, right after a call that leaves NaN in every workgroup's LDS."""
    lens, starts = [130, 64], [0, 5]
    c = lambda *t: [x.to(DEV) for x in t]  # noqa: E731
    nan = _inputs([64] * 16, 128, 1, 128, 64, dtype, "fixed")
    q, k, d, v, beta, state = _inputs(lens, 3, 3, dim, 40, dtype, "token", dim)
    want = ref.gated_state_scan(*(x.double() for x in (q, k, d, v, beta)), _meta(lens, starts, "cpu"), state.double(), False)
    (nq, nk, nd, nv, ns), (q, k, d, v, beta, state) = c(nan[0], nan[1], nan[2], nan[3], nan[5]), c(q, k, d, v, beta, state)
    ops.gated_state_scan(nq, nk, nd, nv, None, _meta([64] * 16, [1] * 16, DEV), ns * math.nan, False)
    got = ops.gated_state_scan(q, k, d, v, beta, _meta(lens, starts, DEV), state, False)
    torch.testing.assert_close(got.cpu().double(), want.double(), rtol=0, atol=1e-5 * (8 + 4 * math.sqrt(130)))


def test_keys_at_the_end_of_their_memory(ops):
    """32 key features leave two of a workgroup's four waves without any: nothing is read past the last key."""
    lens, H, dim, vdim = [64] * 64, 2, 32, 32
    q, k, d, v, beta, state = _inputs(lens, H, H, dim, vdim, torch.bfloat16, "token")
    want = ref.gated_state_scan(*(x.double() for x in (q, k, d, v, beta)), _meta(lens, [0] * 64, "cpu"), state.double(), False)
    whole = torch.empty(12 << 18, device=DEV)     # 12 MiB: a memory block of its own, k its last MiB
    tail = whole[-k.numel():].view(k.shape).copy_(k)
    got = ops.gated_state_scan(q.to(DEV), tail, d.to(DEV), v.to(DEV), beta.to(DEV), _meta(lens, [0] * 64, DEV), state.to(DEV), False)
    torch.testing.assert_close(got.cpu().double(), want.double(), rtol=0, atol=1e-5 * (8 + 4 * math.sqrt(64)))


@pytest.mark.parametrize("decay", ["fixed", "token"])
def test_state_off_16_bytes(ops, decay):
    """A state that does not lie on 16 bytes (a slice of a larger table) goes token by token."""
    lens, starts = [70, 1, 20], [3, 5, 0]
    q, k, d, v, beta, state = _inputs(lens, 3, 1, 5, 7, torch.bfloat16, decay)
    table = torch.cat([state.new_zeros(1), state.flatten()])
    want_state = state.double()
    want = ref.gated_state_scan(q.double(), k.double(), d.double(), v.double(), None if beta is None else beta.double(),
                                _meta(lens, starts, "cpu"), want_state, False)
    c = lambda x: None if x is None else x.to(DEV)  # noqa: E731
    off = c(table)[1:].view(state.shape)
    assert off.data_ptr() % 16 == 4
    got = ops.gated_state_scan(c(q), c(k), c(d), c(v), c(beta), _meta(lens, starts, DEV), off, False)
    bound = 1e-5 * (8 + 4 * math.sqrt(70))
    torch.testing.assert_close(got.cpu().double(), want.double(), rtol=0, atol=bound)
    torch.testing.assert_close(off.cpu().double(), want_state, rtol=0, atol=bound)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,H,dim", [(2, 4, 64), (9, 128, 32), (40, 4, 64), (2, 2, 128), (65, 4, 64), (64, 4, 64)])
def test_segments_around_the_shortest_chunked_one(ops, dtype, n, H, dim):
    """Segments of one token less, as many and one more than the rule's shortest, beside single tokens; 256, 257 and more
    workgroups of 64 columns."""
    from byzantine_consensus_llm_agents_amd.ops.seqstate import chunked_from
    least = chunked_from(n, H, dim, dtype == torch.float32)
    lens = [(least - 1, least, least + 1, 1)[i % 4] for i in range(n)]
    q, k, d, v, beta, state = _inputs(lens, H, 1, dim, 64, dtype, "token", n)
    starts = [i % 3 for i in range(n)]
    want_state = state.double()
    want = ref.gated_state_scan(*(x.double() for x in (q, k, d, v, beta)), _meta(lens, starts, "cpu"), want_state, False)
    got_state, meta = state.to(DEV), _meta(lens, starts, DEV)
    meta.max_q_len = max(lens)
    got = ops.gated_state_scan(*(x.to(DEV) for x in (q, k, d, v, beta)), meta, got_state, False)
    bound = 1e-5 * (8 + 4 * math.sqrt(least))
    torch.testing.assert_close(got.cpu().double(), want.double(), rtol=0, atol=bound)
    torch.testing.assert_close(got_state.cpu().double(), want_state, rtol=0, atol=bound)
