"""Which kernel a recurrence with one decay per head takes (`chunked_from` in ops/seqstate.py), with a library that only
notes its calls: no GPU."""
import types

import pytest
import torch

from byzantine_consensus_llm_agents_amd.models.transformer import AttnMeta
from byzantine_consensus_llm_agents_amd.ops import seqstate


class _Notes:
    def __init__(self):
        self.calls = []

    def bcg_decay_chunks_tokens(self):
        return 64

    def __getattr__(self, name):
        return lambda *a: self.calls.append((name[4:], a)) or 0


def _route(monkeypatch, lens, H, dim, dtype=torch.bfloat16, hint=None, decode=False, delta=False, off=0):
    monkeypatch.setattr(seqstate, "_stream", lambda: 0)
    lib, T, B = _Notes(), sum(lens), len(lens)
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32)  # noqa: E731
    starts = [sum(lens[:i]) for i in range(B + 1)]
    meta = AttnMeta(positions=torch.zeros(T, dtype=torch.int32), slots=None, block_tables=None, seq_lens=i32(*lens), decode=decode,
                    q_start=i32(*starts), state_rows=i32(*range(B)), max_q_len=hint or max(lens), token_seq=torch.zeros(T, dtype=torch.int32))
    q = torch.zeros(T, H, dim)
    state = torch.zeros(B * H * dim * 8 + 4)[off:off + B * H * dim * 8].view(B, H, dim, 8)
    seqstate.seqstate_ops(lib)["gated_state_scan"](q, q, torch.ones(T, H, 1), torch.zeros(T, H * 8, dtype=dtype), torch.ones(T, H), meta, state, delta)
    return [n for n, _ in lib.calls], [a[-3] for n, a in lib.calls if n == "decay_chunks"]


BOTH, ONE = ["decay_chunks", "gated_state_scan"], ["gated_state_scan"]


@pytest.mark.parametrize("lens,H,dim,kw,want,least", [
    ([16], 4, 64, {}, ["decay_chunks"], 16), ([15], 4, 64, {}, ONE, None), ([31], 4, 64, dict(dtype=torch.float32), ONE, None),
    ([24] * 4, 4, 64, {}, ONE, None), ([32] * 4, 4, 64, {}, BOTH, 32), ([16] * 64, 16, 64, {}, BOTH, 16),
    ([16] * 4, 4, 65, {}, BOTH, 16), ([23] * 4, 4, 65, dict(dtype=torch.float32), ONE, None),
    ([16] * 64, 16, 65, dict(dtype=torch.float32), BOTH, 16), ([100] * 64, 2, 32, dict(dtype=torch.float32), ONE, None), ([100] * 63, 2, 32, dict(dtype=torch.float32), BOTH, 48),
    ([3] * 64, 4, 128, {}, ONE, None), ([3] * 64, 4, 128, dict(hint=1), BOTH, 16), ([20] * 4, 4, 64, dict(hint=1), BOTH, 16),   # no word on the longest
    ([200] * 2, 4, 128, dict(decode=True), ONE, None), ([200] * 2, 4, 128, dict(delta=True), ONE, None),
    ([200] * 2, 4, 128, dict(off=1), ONE, None), ([200] * 2, 4, 128, dict(off=4), BOTH, 16)])
def test_route(monkeypatch, lens, H, dim, kw, want, least):
    names, passed = _route(monkeypatch, lens, H, dim, **kw)
    assert names == want and passed == ([] if least is None else [least])
