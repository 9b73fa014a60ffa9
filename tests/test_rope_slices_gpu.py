"""Rotary and cache write of small steps, a token's heads and values over several workgroups.  GPU only."""
import pytest
import torch

import test_row_kernels_gpu as rows

pytestmark = pytest.mark.gpu
ops = rows.ops


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,n_q,n_kv,maps,dim,vdim,rot", [
    (1, 32, 8, 2, 64, 128, 64),      # four slices, values and turned groups in all of them
    (128, 32, 8, 2, 64, 128, 64),    # the last count with four
    (129, 32, 8, 2, 64, 128, 64),    # three
    (257, 20, 2, 1, 52, 20, 12),     # one from 257 on; groups that are not turned
    (170, 19, 3, 1, 128, 100, 128),  # two of three, the last one with a remainder
    (5, 1, 5, 1, 8, 404, 0)])        # slices of values only
def test_a_token_over_several_workgroups(ops, dtype, T, n_q, n_kv, maps, dim, vdim, rot):
    rows.test_rope_tokens_of_a_group(ops, dtype, n_q, n_kv, maps, dim, vdim, rot, T)
