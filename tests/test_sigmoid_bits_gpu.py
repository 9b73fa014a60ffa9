"""Short convolutions and gated head norms in bf16: the fp32 instance's results, rounded once.  The same sums in the same order, so the same bits;
a sigmoid of fewer bits shows where a value lies next to the middle of two.  GPU only."""
import pytest
import torch

from test_decay_chunks_gpu import _meta
from test_row_kernels_gpu import ops  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [[700, 300], [3000]])   # (a row a workgroup, runs of rows)
def test_short_conv(ops, lens):
    torch.manual_seed(1)
    T, C, taps = sum(lens), 2048, 4
    meta = _meta(lens, [0] * len(lens), "cuda")
    y = (3.0 * torch.randn(T, C, device="cuda")).to(torch.bfloat16)
    w, b = torch.randn(C, taps, device="cuda"), torch.randn(C, device="cuda")
    state = torch.zeros(len(lens) + 1, taps - 1, C, device="cuda", dtype=torch.bfloat16)
    got = ops.short_conv(y, C, w, meta, state.clone(), "silu", b)
    want = ops.short_conv(y.float(), C, w, meta, state.float(), "silu", b).to(torch.bfloat16)
    assert torch.equal(got, want), (got != want).sum()


@pytest.mark.parametrize("act", ["sigmoid", "silu"])
def test_head_norm_gate(ops, act):
    torch.manual_seed(2)
    T, H, dim = 1500, 16, 128
    o = torch.randn(T, H, dim, device="cuda")
    w = torch.randn(dim, device="cuda")
    gate = (3.0 * torch.randn(T, H * dim, device="cuda")).to(torch.bfloat16)
    got = ops.head_norm_gate(o, w, 1e-5, gate, torch.bfloat16, act)
    want = ops.head_norm_gate(o, w, 1e-5, gate.float(), torch.float32, act).to(torch.bfloat16)
    assert torch.equal(got, want), (got != want).sum()
