"""Row kernels of the decoders at the edges of their variants (threads of a row, vectors of a thread) against the reference ops.  GPU only.
Bounds: fp32 sums in another order, one rounding to bf16 (2^-8); fp8 rows match up to single values that round the other way."""
import pytest
import torch

import test_kernels_gpu as kernels
from byzantine_consensus_llm_agents_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
hip = kernels.hip

ROWS = [1, 256, 257]                                                # a row per workgroup of one vector a thread, and more of them
WIDTHS = [8, 2048, 2056, 4096, 4104, 6144, 6152, 8192]


@pytest.mark.parametrize("T", ROWS)
@pytest.mark.parametrize("H", WIDTHS)
def test_norms(hip, T, H):
    x, res = torch.randn(T, H, device="cuda").bfloat16(), torch.randn(T, H, device="cuda").bfloat16()
    w = (1 + 0.1 * torch.randn(H, device="cuda")).bfloat16()
    table, tokens = torch.randn(9, H, device="cuda").bfloat16(), torch.randint(0, 9, (T,), device="cuda", dtype=torch.int32)
    for (y, r), (yr, rr) in ((hip.add_rmsnorm(x, res.clone(), w, 1e-6), ref.add_rmsnorm(x, res.clone(), w, 1e-6)),
                             (hip.add_rmsnorm(x, None, w, 1e-6), ref.add_rmsnorm(x, None, w, 1e-6)),
                             ((hip.rmsnorm(x, w, 1e-6), x), (ref.rmsnorm(x, w, 1e-6), x)),
                             (hip.embed_rmsnorm(tokens, table, w, 1e-6), ref.add_rmsnorm(table[tokens.long()], None, w, 1e-6))):
        assert torch.equal(r, rr)
        torch.testing.assert_close(y, yr, rtol=2 ** -7, atol=1e-5)
    kernels._fp8_close(*hip.rmsnorm_fp8(x, w, 1e-6), *ref.quant_fp8(ref.rmsnorm(x, w, 1e-6)))
