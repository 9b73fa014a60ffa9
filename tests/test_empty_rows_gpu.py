"""Row kernels over rows of no columns: nothing is read, the results are empty.  GPU only."""
import pytest
import torch

from test_row_kernels_gpu import ops  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [3, 300])
def test_no_columns(ops, T):
    bf16 = dict(device="cuda", dtype=torch.bfloat16)
    x, w, table = torch.empty(T, 0, **bf16), torch.empty(0, **bf16), torch.empty(9, 0, **bf16)
    tokens = torch.zeros(T, device="cuda", dtype=torch.int32)
    assert ops.rmsnorm(x, w, 1e-5).shape == (T, 0)
    assert ops.add_rmsnorm(x, torch.empty_like(x), w, 1e-5)[0].shape == (T, 0)
    assert ops.embed_rmsnorm(tokens, table, w, 1e-5)[1].shape == (T, 0)
    for q, s in (ops.rmsnorm_fp8(x, w, 1e-5), ops.add_rmsnorm_fp8(x, None, w, 1e-5)[:2], ops.embed_rmsnorm_fp8(tokens, table, w, 1e-5)[:2]):
        assert q.shape == (T, 0)
        torch.testing.assert_close(s, torch.full_like(s, 1e-12 / 448.0), rtol=1e-6, atol=0)
    for dtype in (torch.bfloat16, torch.float32):
        parts = [torch.empty(T, 0, device="cuda", dtype=dtype)] * 2
        y = ops.residual_add_rmsnorm32(torch.empty(T, 0, device="cuda"), parts, torch.empty(0, device="cuda"), 1e-5, 1.0, dtype)
        assert y.shape == (T, 0)
    torch.cuda.synchronize()
