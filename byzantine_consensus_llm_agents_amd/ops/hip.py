"""ctypes bindings of ``libbcg_kernels.so`` (csrc/kernels, gfx950).

Every wrapper validates dtypes, contiguity and shapes on the host before it
launches (a kernel that indexes out of bounds can take down every GPU of the
node), then launches on the current HIP stream -- so the calls are captured
by ``torch.cuda.graph`` like any PyTorch op.  A missing library raises: with a
GPU the engine never silently falls back to the PyTorch references.
"""

import ctypes
import os
from types import SimpleNamespace

import torch

from ..utils.build import kernel_sources, kernels_source_hash, kernels_target
from .operands import bare, watched

_LIB = None
# Rows per prefill attention tile unless BCG_PREFILL_TILE_ROWS says otherwise (prefill_tile_rows)
PREFILL_TILE_ROWS = 128
PREFILL32_MAX_BLOCKS = 1024  # csrc/kernels/attention.hip: the 32x32 kernel's LDS block-id table

# csrc/kernels/gemm_skinny.hip: most rows, most rows with a fused norm, longest rows in bytes
SKINNY_ROWS, SKINNY_NORM_ROWS, SKINNY_ROW_BYTES = 64, 16, 65536
MID_ROWS = 1536  # csrc/kernels/gemm_mid.hip: most rows
SKINNY_LONG_K = 12288  # past it: fewer shapes gain (`few_rows_pay`), logged apart

c_int, c_float, c_void_p, c_uint32, c_int64 = ctypes.c_int, ctypes.c_float, ctypes.c_void_p, ctypes.c_uint32, ctypes.c_int64


class StaleLibraryError(RuntimeError):
    pass


def library_stamp(lib: ctypes.CDLL) -> str:
    fn = getattr(lib, "bcg_source_hash", None)
    if fn is None:
        return None
    fn.argtypes, fn.restype = [], ctypes.c_char_p
    return fn().decode()


def check_source_stamp(lib: ctypes.CDLL, path: str):
    """Refuse a library built from other sources than the tree's csrc/kernels.

    ``utils/build.py`` stamps the library with a hash of every kernel source.
    A deployment without sources (no csrc/kernels) has nothing to compare with
    and is accepted."""
    if not kernel_sources()[0]:
        return
    want, got = kernels_source_hash(), library_stamp(lib)
    if got != want:
        raise StaleLibraryError(
            f"{path} was built from other sources (stamp {got!r}, csrc/kernels {want!r}); rebuild with "
            "`python -m byzantine_consensus_llm_agents_amd.utils.build --force`")


def few_rows_stay(M: int, N: int, K: int, gated: bool) -> bool:
    """33 to 64 rows that the few-row kernel takes (`few_rows_pay`) and the one-round kernel could: whether the first keeps them.

    Times of the one-round kernel over the few-row kernel's at 1018 products of 2.7 M elements of W and more: 0.84 on average, 34 of 1.03 to 1.14, most of
    them where its plan is 48 x 32 tiles in one part that leave a quarter of the CUs idle and the few-row kernel's rows are whole turns: up to
    48 rows, K in steps of 512 from 2048 to 4096, 4097 to 6500 columns (gated 2700 to 6500) 1.01 on average, up to 1.14 (44 rows, 6144 x 4096:
    16.1 us for 17.5).  14 of the others are 1.03 to 1.07 slower.  Smaller W: 0.77 to 0.82, a gain that
    this line still leaves to the few-row kernel."""
    if N * K < 2700000:
        return True
    return M <= 48 and K % 512 == 0 and 2048 <= K <= 4096 and (2700 if gated else 4097) <= N <= 6500


def load_library(path: str = None) -> ctypes.CDLL:
    global _LIB
    if _LIB is not None:
        return _LIB
    path = path or os.environ.get("BCG_KERNELS_LIB") or kernels_target()  # override: variant builds (tools)
    if not os.path.exists(path):
        raise RuntimeError(f"HIP kernel library not found at {path}; run `python -m "
                           "byzantine_consensus_llm_agents_amd.utils.build` (hipcc --offload-arch=gfx950)")
    lib = ctypes.CDLL(path)
    check_source_stamp(lib, path)
    sig = {
        "bcg_add_rmsnorm": [c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_float, c_int, c_void_p],
        "bcg_silu_mul": [c_void_p, c_void_p, c_int64, c_int, c_void_p],
        "bcg_embed_rmsnorm": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_float, c_void_p],
        "bcg_qk_norm_rope_kv_write": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                      c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_int,
                                      c_float, c_int, c_int, c_void_p],
        "bcg_paged_attention_decode": [c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_void_p, c_int,
                                       c_void_p, c_int, c_int, c_int, c_int, c_float, c_void_p, c_int,
                                       c_int, c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_int, c_void_p,
                                       c_int, c_void_p, c_void_p, c_int, c_int, c_void_p],
        "bcg_paged_attention_prefill": [c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_void_p, c_int,
                                        c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_float,
                                        c_void_p, c_int, c_int, c_void_p],
        "bcg_paged_attention_prefill32": [c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_void_p, c_int,
                                          c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_float,
                                          c_void_p, c_int, c_int, c_void_p],
        "bcg_decode_split_tokens": [c_int, c_int, c_int],
        "bcg_decode_max_splits": [c_int, c_int],
        "bcg_decode_max_context": [c_int],
        "bcg_quant_fp8": [c_void_p, c_void_p, c_void_p, c_int, c_int, c_void_p],
        "bcg_add_rmsnorm_fp8": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_float, c_int,
                                c_void_p],
        "bcg_silu_mul_fp8": [c_void_p, c_void_p, c_void_p, c_int, c_int, c_void_p],
        "bcg_embed_rmsnorm_fp8": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_float,
                                  c_void_p],
        "bcg_gemm_nt": [c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                        c_int, c_int, c_int, c_int, c_int, c_void_p],
        "bcg_gemm_nt_fp8": [c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                            c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_void_p],
        "bcg_decode_pairs": [c_void_p] * 6 + [c_float, c_void_p, c_void_p, c_int, c_int, c_int, c_void_p, c_int, c_void_p, c_int,
                             c_int, c_int, c_int, c_float, c_int, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p],
        "bcg_decode_order": [c_void_p, c_int, c_void_p, c_void_p],
        "bcg_gemm_skinny": [c_int, c_void_p, c_void_p, c_void_p, c_float, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int,
                            c_void_p],
        "bcg_gemm_skinny_fp8": [c_int] + [c_void_p] * 7 + [c_int] * 3 + [c_void_p],
        "bcg_capture_id": [c_void_p],
        "bcg_gemm_mid_plan": [c_int] * 5,
        "bcg_gemm_mid_parts": [c_int] * 4 + [ctypes.POINTER(c_int)],
        "bcg_gemm_mid": [c_int, c_int] + [c_void_p] * 9 + [c_int] * 4 + [c_void_p],
        "bcg_gemm_mid_act": [c_int] + [c_void_p] * 7 + [c_int] * 6 + [c_void_p],
        "bcg_gemm_tile": [c_int, ctypes.POINTER(c_int), ctypes.POINTER(c_int)],
        "bcg_gemm_num_cfgs": [],
        "bcg_embed_scale_rmsnorm": [c_void_p, c_void_p, c_float, c_void_p, c_void_p, c_float, c_float, c_void_p, c_void_p,
                                    c_int, c_int, c_int, c_int, c_void_p],
        "bcg_residual_add_rmsnorm32": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_float,
                                       c_float, c_void_p, c_int, c_int, c_int, c_void_p],
        "bcg_act_fn": [c_void_p, c_void_p, c_int64, c_int, c_int64, c_int, c_int, c_void_p],
        "bcg_rope_multi_kv_write": [c_void_p, c_int64, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p,
                                    c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p],
        "bcg_multimap_split_keys": [],
        "bcg_multimap_pairs": [c_int] * 5,
        "bcg_multimap_attention": [c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p,
                                   c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int,
                                   c_float, c_float, c_float, c_float, c_int, c_int, c_int, c_int, c_void_p, c_float,
                                   c_void_p, c_int, c_int, c_int, c_int, c_int, c_void_p, c_void_p],
        "bcg_embed_position": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int,
                               c_int, c_void_p],
        "bcg_residual_rms_norm": [c_void_p, c_void_p, c_int, c_void_p, c_float, c_void_p, c_void_p, c_void_p, c_int, c_int,
                                  c_void_p, c_float, c_void_p, c_int, c_int, c_int, c_void_p],
        "bcg_retention_prepare": [c_void_p, c_int64, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_int, c_float, c_float,
                                  c_void_p, c_void_p, c_int, c_int, c_void_p],
        "bcg_residual_layer_norm": [c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_float, c_int, c_void_p, c_void_p,
                                    c_float, c_void_p, c_int, c_int, c_int, c_void_p],
        "bcg_embed_hashed_bigram": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_float,
                                    c_void_p, c_int, c_int, c_int, c_float, c_float, c_float, c_void_p, c_void_p, c_void_p,
                                    c_int, c_int, c_int, c_int, c_int, c_void_p],
        "bcg_residual_mix_norm": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_float, c_float,
                                  c_float, c_float, c_float, c_void_p, c_void_p, c_int, c_int, c_int, c_void_p],
        "bcg_short_conv": [c_void_p, c_int64, c_int, c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                           c_int, c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_void_p],
        "bcg_rope_pairs_kv_write": [c_void_p, c_int64, c_void_p, c_void_p, c_void_p, c_void_p, c_float, c_void_p, c_int,
                                    c_float, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int,
                                    c_float, c_int, c_int, c_int, c_int, c_void_p],
        "bcg_rotate_pairs": [c_void_p, c_void_p, c_void_p, c_float, c_void_p, c_int, c_int, c_int, c_int, c_void_p],
        "bcg_hgrn2_prepare": [c_void_p, c_int64, c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int,
                              c_int, c_int, c_void_p],
        "bcg_delta_prepare": [c_void_p, c_int64, c_void_p, c_int64, c_int, c_void_p, c_int64, c_int, c_void_p, c_void_p,
                              c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_void_p],
        "bcg_gated_state_scan": [c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p, c_void_p, c_void_p, c_void_p,
                                 c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int,
                                 c_int, c_int, c_void_p],
        "bcg_decay_chunks_tokens": [],
        "bcg_decay_chunks": [c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_int64, c_void_p, c_void_p, c_void_p, c_void_p,
                             c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p],
        "bcg_head_norm_gate": [c_void_p, c_void_p, c_float, c_void_p, c_int64, c_void_p, c_int, c_int, c_int, c_int, c_void_p,
                               c_int, c_int, c_void_p],
        "bcg_hyper_embed_norm": [c_void_p, c_void_p, c_void_p, c_void_p, c_float, c_void_p, c_void_p, c_int, c_int, c_int,
                                 c_int, c_int, c_void_p],
        "bcg_hyper_update_norm": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_float, c_void_p,
                                  c_int, c_int, c_int, c_int, c_void_p],
        "bcg_rope_norm_kv_write": [c_void_p, c_int64, c_void_p, c_void_p, c_void_p, c_int, c_float, c_void_p, c_int64,
                                   c_float, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_int,
                                   c_int, c_void_p],
        "bcg_exp_gate_prepare": [c_void_p, c_int64, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_float, c_float,
                                 c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_void_p,
                                 c_void_p, c_int, c_int, c_int, c_int, c_int, c_void_p],
        "bcg_softcap": [c_void_p, c_int64, c_float, c_void_p],
        "bcg_moe_route_scored": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int,
                                 c_float, c_int, c_void_p],
        "bcg_embed_scale_dyt": [c_void_p, c_void_p, c_float, c_float, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int,
                                c_int, c_int, c_void_p],
        "bcg_residual_post_norm": [c_void_p, c_void_p, c_int, c_int, c_float, c_void_p, c_void_p, c_float, c_int, c_float,
                                   c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_void_p],
        "bcg_rmsnorm_cols": [c_void_p, c_int64, c_int, c_int, c_void_p, c_float, c_void_p, c_int, c_int, c_void_p],
        "bcg_latent_kv_write": [c_void_p, c_int64, c_int, c_int, c_int, c_void_p, c_float, c_void_p, c_void_p, c_void_p,
                                c_int, c_float, c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_void_p],
        "bcg_rope_tail": [c_void_p, c_int, c_int, c_void_p, c_int, c_int, c_void_p, c_void_p, c_int, c_float, c_int, c_int,
                          c_int, c_int, c_void_p],
        "bcg_head_linear": [c_void_p, c_int64, c_int64, c_void_p, c_void_p, c_int64, c_int64] + [c_int] * 4 + [c_void_p, c_void_p]
        + [c_int] * 3 + [c_float, c_void_p, c_int64, c_int, c_void_p],
        "bcg_gate_mul": [c_void_p, c_void_p, c_int64, c_void_p, c_int64, c_int, c_int, c_int, c_int, c_void_p],
        "bcg_gemm_w4_act": [c_int] + [c_void_p] * 4 + [c_int] * 4 + [c_float, c_void_p],
        "bcg_gated_act": [c_void_p, c_void_p, c_int64, c_int, c_int, c_float, c_int, c_void_p],
        "bcg_ssm_prepare": [c_void_p, c_int64, c_int, c_void_p, c_int64, c_int, c_void_p, c_void_p, c_void_p, c_void_p,
                            c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_void_p],
        "bcg_gated_group_norm": [c_void_p, c_void_p, c_int64, c_void_p, c_void_p, c_int64, c_void_p, c_float, c_void_p,
                                 c_int, c_int, c_int, c_int, c_int, c_void_p],
        "bcg_gelu_gather_mul": [c_void_p, c_void_p, c_void_p, c_int64, c_int, c_void_p, c_int64, c_int, c_int, c_int,
                                c_void_p],
        "bcg_moe_tile_rows": [],
        "bcg_moe_route": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int,
                          c_int, c_int, c_void_p],
        "bcg_moe_align": [c_void_p, c_int, c_int, c_void_p, c_int, c_void_p, c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int,
                          c_int, c_void_p],
        "bcg_experts_post_norm": [c_void_p] * 4 + [c_int] * 3 + [c_float, c_void_p, c_void_p, c_float, c_int, c_float] + [c_void_p] * 3
        + [c_int, c_int, c_void_p],
        "bcg_gemm_w4_grouped": [c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_float, c_void_p, c_int,
                                c_int, c_void_p],
        "bcg_moe_route_table": [c_void_p, c_void_p] + [c_int] * 4 + [c_void_p] * 3,
        "bcg_moe_rows_tile": [],
        "bcg_moe_rows": [c_void_p, c_int64, c_int64, c_void_p, c_void_p, c_int64, c_void_p, c_void_p] + [c_int] * 8
                        + [c_float, c_void_p],
        "bcg_moe_gemm": [c_void_p, c_int64, c_void_p, c_void_p, c_int64, c_void_p, c_void_p, c_int, c_int, c_int,
                         c_int, c_int, c_int, c_int, c_float, c_int, c_void_p],
        "bcg_moe_combine": [c_void_p] * 4 + [c_int, c_void_p] + [c_int] * 4 + [c_void_p],
        "bcg_guided_sample": [c_void_p, c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                              c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p,
                              c_uint32, c_int, c_int, c_int, c_int, c_void_p],
    }
    for name, argtypes in sig.items():
        fn = getattr(lib, name)
        fn.argtypes = argtypes
        fn.restype = c_int64 if name in ("bcg_gemm_mid_parts", "bcg_capture_id") else c_int
    _LIB = lib
    return lib


def _stream() -> int:
    return torch.cuda.current_stream().cuda_stream


def _p(t: torch.Tensor):
    return ctypes.c_void_p(t.data_ptr())


def _check(rc: int, name: str):
    if rc != 0:
        raise RuntimeError(f"{name} launch failed (rc={rc})")


def _req(cond: bool, msg: str):
    if not cond:
        raise ValueError(msg)


def _kv_fp8(k_cache: torch.Tensor, v_cache: torch.Tensor) -> int:
    """1 for an fp8 (e4m3fn) KV cache, 0 for bf16; anything else is refused before launch."""
    _req(k_cache.dtype == v_cache.dtype and k_cache.dtype in (torch.bfloat16, torch.float8_e4m3fn)
         and k_cache.is_contiguous() and v_cache.is_contiguous(), "KV cache: contiguous bf16 or float8_e4m3fn")
    return int(k_cache.dtype == torch.float8_e4m3fn)


def few_rows_pay(M: int, N: int, row_bytes: int, gated: bool) -> bool:
    """Whether M <= SKINNY_ROWS rows of bf16 gain by the few-row kernel, W of N rows of row_bytes; gated: the [gate; up] form, which saves the
    other side a pass over the product.

    Each CU reads all of X for its N / 256 rows of W, so few long rows of W lose to a split of K over the CUs; a turn of a workgroup's
    waves is 2048 bytes of a row, so rows of one and a half turns leave waves idle; from 33 rows on one pass over W only.  Times of this kernel
    over those of tile kernels or library (which has a kernel for exactly 32 rows); "but" is what the lines leave to them:
    * up to 16 rows 0.22 to 1.0 (to 1.1 for one or two rows of up to 1024 x 12288); but 13312 to 16384 long, few of them: 256 1.11 to
      1.68, with 13 rows and more 512 and 1024 1.02 to 1.13; gated, up to 3072 of them 1.05 to 1.17 against the plain form and a pass;
    * 17 to 32 rows, up to 8192 bytes 0.45 to 1.03, longer ones from 4096 of them on 0.33 to 1.03; but up to 31 rows 512 x 640 to 512 x 896 1.04 to 1.18, 256 x 1536 1.13 to
      1.22, exactly 32 rows up to 2048 x 2560 and 1536 x 3584 0.98 to 1.17, up to 1024 x 3072 or x 4096 0.98 to 1.19;
    * 33 to 48 rows 0.46 to 1.06; but up to 1024 x 448, 640 x 640 and 512 x 768 1.02 to 1.17, 3072 x 1536 1.01 to 1.13, 256 x 1536 1.5, 2048 x 2560 1.09 to 1.39, 1536 x
      3072 1.17 to 1.26, 8192 x 4096 1.03 to 1.06, longer rows 1.3 and more;
    * 49 to 64 rows 0.62 to 1.10, with 1024 to 2048 x 2048 1.02 to 1.16 (a store; gated 0.87 to 0.92); but 1024 x 448 1.05 to 1.27, 6144 x 448 1.04 to
      1.16, 3072 x 1536 1.14 to 1.26, 4096 x 4096 1.08;
    * gated 0.42 to 1.03; but with 33 to 48 rows 256 x 1536 1.09, 2048 x 2560 1.08 to 1.1, and the longer rows of the lines above."""
    part = row_bytes % 2048 != 0     # the last turn is not a whole one
    if M <= 16:
        if gated or row_bytes <= 2 * SKINNY_LONG_K:
            return row_bytes <= 2 * SKINNY_LONG_K or N >= 4096
        return row_bytes > 32768 or N >= (1536 if M > 12 else 512 if row_bytes <= 28672 else 384)
    if M <= 32:
        if gated or row_bytes > 8192:
            return row_bytes <= 8192 or N >= 4096
        if row_bytes > 4096:
            return not (M == 32 and N <= (2048 if part and row_bytes <= 6144 else 1024))
        if row_bytes > 2048:
            return not part or N > 256
        return not (1024 < row_bytes < 2048 and 256 < N <= 512 and M < 32)
    if N > 32 * 256 or row_bytes > (8192 if M <= 48 else 4096):
        return False
    if M <= 48:
        if gated and part:
            return not 1024 < N < 3072 if row_bytes > 4096 else row_bytes < 2048 or N >= 512
        if gated or row_bytes == 2048:
            return True
        if row_bytes > 4096:
            return N >= 3072 if part else N >= 2048 if row_bytes <= 6144 else N <= 6144
        if row_bytes > 2048:
            return not part or N >= 4096
        return N <= 256 or row_bytes >= 1792 or N >= (1536 if row_bytes < 1024 else 768 if row_bytes < 1536 else 640)
    if gated or 1536 <= row_bytes <= 2048:
        return N >= 1024
    if row_bytes < 1536:
        return (1536 if row_bytes < 1024 else 1024) <= N <= 4096
    return N >= (4096 if part else 1024)


def part_rule(pairs: int, chunk: int, chunks: int):
    """(parts, one, each, ways, extra) of `PartRule` in csrc/kernels/common.h for `pairs` pairs of a decode step whose block table has room for `chunks`
    chunks of 32 keys, `chunk` bytes of K and V each (the contexts themselves are on the device).

    Rows stay whole up to 448 KB of K/V of a pair (heads of 128, us for 1, 2, 3, 4, 8 parts and a merge launch: 80 pairs of 400 tokens 9.4, 12.3, 12.5, of 1000 19.5, 17.9,
    16.7, of 2500 38.6, 29.1, 27.3; 8 pairs of 400 8.1, 9.8, 10, 9.5, of 1000 11, 11.8, 11.5, 10.4, 10.1, of 6000 36, 24, 20, 16.7, 13.5), up to 2 MB where
    the pairs fill the CUs by themselves (160 pairs of 1000 22.8, 28.6): there it is for rows that are long beside the others, 25 us by one workgroup, and with
    448 KB the look over the rows cost steps of equal ones 2 to 4 % (808 pairs of 1000 tokens 82.5, 85.7).  257 to 352 pairs leave most CUs with one and some
    with two: cut among 1024 workgroups they even out (320 pairs of 5000 tokens 183 -> 162, 264 of 2000 63 -> 60.5; 384 of 5000 192, 193, 400 194, 197)."""
    few, uneven = pairs <= 128, 256 < pairs <= 352
    one, each = (448 if few or uneven else 2048) * 1024 // chunk, max(1, 128 * 1024 // chunk)
    ways = 1024 if uneven else 256
    parts = min(16, -(-chunks // each)) if chunks > one else 1
    return parts, one, each, ways, min(ways, pairs * (parts - 1))


def hip_ops() -> SimpleNamespace:
    lib = load_library()

    def add_rmsnorm(x, residual, w, eps):
        _req(x.dtype == torch.bfloat16 and x.is_contiguous() and x.dim() == 2, "add_rmsnorm: x bf16 [T,H]")
        T, H = x.shape
        _req(w.shape == (H,) and w.dtype == torch.bfloat16, "add_rmsnorm: weight [H] bf16")
        has_res = residual is not None
        if not has_res:
            residual = torch.empty_like(x)
        else:
            _req(residual.shape == x.shape and residual.is_contiguous(), "add_rmsnorm: residual shape")
        out = torch.empty_like(x)
        _check(lib.bcg_add_rmsnorm(_p(x), _p(residual), _p(w), _p(out), T, H, eps, int(has_res), _stream()),
               "add_rmsnorm")
        return out, residual

    def embed_rmsnorm(tokens, table, w, eps):
        """(rmsnorm(table[tokens]) * w, table[tokens]) in one pass over the gathered rows."""
        _req(tokens.dtype == torch.int32 and tokens.is_contiguous() and tokens.dim() == 1, "tokens int32 [T]")
        _req(table.dtype == torch.bfloat16 and table.is_contiguous() and table.dim() == 2, "table bf16 [V,H]")
        T, H = tokens.numel(), table.shape[1]
        _req(w.shape == (H,) and w.dtype == torch.bfloat16, "embed_rmsnorm: weight [H] bf16")
        residual = torch.empty(T, H, dtype=table.dtype, device=table.device)
        out = torch.empty_like(residual)
        _check(lib.bcg_embed_rmsnorm(_p(tokens), _p(table), _p(w), _p(residual), _p(out), T, H, eps, _stream()),
               "embed_rmsnorm")
        return out, residual

    def rmsnorm(x, w, eps):
        """Plain RMSNorm (mode 2: the residual stream is not touched)."""
        _req(x.dtype == torch.bfloat16 and x.is_contiguous() and x.dim() == 2, "rmsnorm: x bf16 [T,H]")
        T, H = x.shape
        _req(w.shape == (H,) and w.dtype == torch.bfloat16, "rmsnorm: weight [H] bf16")
        out = torch.empty_like(x)
        _check(lib.bcg_add_rmsnorm(_p(x), None, _p(w), _p(out), T, H, eps, 2, _stream()), "rmsnorm")
        return out

    def silu_mul(gu):
        _req(gu.dtype == torch.bfloat16 and gu.is_contiguous() and gu.dim() == 2, "silu_mul: bf16 [T,2I]")
        T, I2 = gu.shape
        out = torch.empty(T, I2 // 2, dtype=gu.dtype, device=gu.device)
        _check(lib.bcg_silu_mul(_p(gu), _p(out), T, I2 // 2, _stream()), "silu_mul")
        return out

    def qk_norm_rope_kv_write(qkv, positions, slots, n_q, n_kv, head_dim, q_norm, k_norm, eps, cos_sin,
                              k_cache, v_cache, layer, contiguous=True):
        """contiguous: the tokens come in runs of consecutive slots (prefill chunks), so V can be
        written a whole KV block at a time; False for decode batches (one token per sequence)."""
        T = qkv.shape[0]
        _req(qkv.is_contiguous() and qkv.shape[1] == (n_q + 2 * n_kv) * head_dim, "qkv shape")
        _req(positions.dtype == torch.int32 and slots.dtype == torch.int32 and positions.numel() == T
             and slots.numel() == T, "positions/slots int32 [T]")
        _req(cos_sin.dtype == torch.float32 and cos_sin.shape[1] == head_dim, "cos_sin table")
        L, NB, nkv_c, BS, hd = k_cache.shape
        _req(nkv_c == n_kv and hd == head_dim and v_cache.shape == (L, NB, n_kv, hd, BS), "kv cache layout")
        q = torch.empty(T, n_q, head_dim, dtype=qkv.dtype, device=qkv.device)
        _check(lib.bcg_qk_norm_rope_kv_write(
            _p(qkv), _p(positions), _p(slots), _p(q), _p(q_norm) if q_norm is not None else None,
            _p(k_norm) if k_norm is not None else None, _p(cos_sin), _p(k_cache), _p(v_cache), layer, T,
            n_q, n_kv, head_dim, NB, BS, eps, _kv_fp8(k_cache, v_cache), int(bool(contiguous)), _stream()),
            "qk_norm_rope_kv_write")
        return q

    def decode_workspace_numel(B, n_q, hd, max_blocks, block_size=16, cascade=True):
        """fp32 split partials (o, m, l) of the flash-decoding split-K (+ the shared-prefix
        pass's slots when `cascade`)."""
        max_splits = lib.bcg_decode_max_splits(max_blocks * block_size, int(cascade))
        return B * n_q * max_splits * (hd + 2)

    def paged_attention_decode(q, k_cache, v_cache, layer, block_tables, seq_lens, scale, workspace=None,
                               cascade=None):
        """`workspace`: optional fp32 split-K scratch of >= decode_workspace_numel(...) elements,
        shared by every decode graph (it is dead between launches) instead of one per graph.
        `cascade`: optional shared-prefix tables (``engine/cascade.py`` ``CascadeTables``):
        rows whose leading KV blocks are shared read them once per group."""
        B, n_q, hd = q.shape
        L, NB, n_kv, BS, _ = k_cache.shape
        _req(q.is_contiguous() and block_tables.dtype == torch.int32 and block_tables.is_contiguous()
             and block_tables.shape[0] == B and seq_lens.numel() == B, "decode attention inputs")
        max_blocks = block_tables.shape[1]
        _req(B <= 2048, "decode attention: at most 2048 rows")
        split = lib.bcg_decode_split_tokens(B, n_kv, max_blocks * BS)
        max_splits = lib.bcg_decode_max_splits(max_blocks * BS, int(cascade is not None))
        need = B * n_q * max_splits * (hd + 2)
        if workspace is None:
            ws = torch.empty(need, dtype=torch.float32, device=q.device)
        else:
            _req(workspace.dtype == torch.float32 and workspace.is_contiguous() and workspace.numel() >= need,
                 "decode attention workspace too small")
            ws = workspace
        cas = [None, None, None, 0, None, 0, None, None, 0, 32]
        if cascade is not None:
            c = cascade
            i32 = torch.int32
            for t in (c.kv_begin, c.split_base, c.grp_rows, c.grp_desc, c.items, c.n_items):
                _req(t.dtype == i32 and t.is_contiguous() and t.device == q.device, "cascade tables: int32 on device")
            _req(c.kv_begin.numel() >= B and c.split_base.numel() >= B, "cascade tables: one entry per row")
            _req(c.grp_desc.dim() == 2 and c.grp_desc.shape[1] == 4 and c.items.dim() == 2 and c.items.shape[1] == 4
                 and c.n_items.numel() >= 1, "cascade tables: grp_desc [G, 4], items [I, 4], n_items [1]")
            cas = [_p(c.kv_begin), _p(c.split_base), _p(c.grp_rows), c.grp_rows.numel(), _p(c.grp_desc),
                   c.grp_desc.shape[0], _p(c.items), _p(c.n_items), c.items.shape[0], c.split_tokens]
        out = torch.empty(B, n_q * hd, dtype=q.dtype, device=q.device)
        _check(lib.bcg_paged_attention_decode(
            _p(q), _p(k_cache), _p(v_cache), layer, NB, n_kv, _p(block_tables), max_blocks, _p(seq_lens),
            B, n_q, hd, BS, scale, _p(ws), max_splits, split, _p(out), _kv_fp8(k_cache, v_cache), *cas,
            _stream()), "paged_attention_decode")
        return out

    def decode_attention_pairs(qkv, positions, slots, n_q, n_kv, hd, q_norm, k_norm, eps, cos_sin, k_cache, v_cache, layer,
                               block_tables, seq_lens, scale, workspace=None, parts=None, order=None):
        """paged_attention_decode(qk_norm_rope_kv_write(...)) for one new token per row of a bf16 cache with heads of 64 or 128, in one launch.
        Rows are different sequences: no row sees what another one stores in this call.  A workgroup for a (row, kv head) pair, several for
        one of a long row (`part_rule`; parts: that many for every one), which meet in `workspace` where it has the room.  order:
        `decode_order` of seq_lens, the pairs' order over the launch."""
        B = qkv.shape[0]
        L, NB, nkv_c, BS, hdc = k_cache.shape
        _req(qkv.dtype == torch.bfloat16 and qkv.is_contiguous() and qkv.shape[1] == (n_q + 2 * n_kv) * hd, "decode qkv")
        _req(nkv_c == n_kv and hdc == hd and hd in (64, 128) and BS == 16 and v_cache.shape == (L, NB, n_kv, hd, BS)
             and not _kv_fp8(k_cache, v_cache), "decode kv cache layout")
        _req(all(t.dtype == torch.int32 and t.is_contiguous() for t in (positions, slots, seq_lens, block_tables))
             and positions.numel() == slots.numel() == seq_lens.numel() == B and block_tables.shape[0] == B, "decode tables")
        _req(order is None or (order.dtype == torch.int32 and order.is_contiguous() and order.numel() == B and order.device == qkv.device), "decode order")
        _req(cos_sin.dtype == torch.float32 and cos_sin.shape[1] == hd and B <= 2048, "decode cos_sin / rows")
        if parts is None:
            rule = part_rule(B * n_kv, 128 * hd, -(-block_tables.shape[1] // 2))
        else:
            rule = (parts, 0, 0, 0, B * n_kv * (parts - 1))
            _req(1 <= parts <= 64 and rule[4] <= 1 << 16, "decode parts")
        need = 2 * rule[4] * (n_q // n_kv) * (hd + 2)
        if workspace is not None:
            _req(workspace.dtype == torch.float32 and workspace.is_contiguous(), "decode attention workspace")
        if need and (workspace is None or workspace.numel() < need):
            workspace = torch.empty(need, dtype=torch.float32, device=qkv.device)
        out = torch.empty(B, n_q * hd, dtype=qkv.dtype, device=qkv.device)
        _check(lib.bcg_decode_pairs(
            _p(qkv), _p(positions), _p(slots), None if q_norm is None else _p(q_norm), None if k_norm is None else _p(k_norm),
            _p(cos_sin), eps, _p(k_cache), _p(v_cache), layer, NB, n_kv, _p(block_tables), block_tables.shape[1], _p(seq_lens), B, n_q, hd,
            BS, scale, *rule, _p(workspace) if need else None, _p(_counters(qkv.device)) if need else None, _p(out),
            None if order is None else _p(order), _stream()), "decode_attention_pairs")
        return out

    def decode_order(seq_lens):
        """The rows of a decode step, longest context first (int32): one launch for all layers' `decode_attention_pairs`."""
        _req(seq_lens.dtype == torch.int32 and seq_lens.is_contiguous() and 0 < seq_lens.numel() <= 2048, "decode order: seq_lens int32 [B]")
        order = torch.empty_like(seq_lens)
        _check(lib.bcg_decode_order(_p(seq_lens), seq_lens.numel(), _p(order), _stream()), "decode_order")
        return order

    def paged_attention_prefill(q, k_cache, v_cache, layer, block_tables, q_start, seq_lens, scale,
                                max_q_len=None, tiles=None, tile_rows=64):
        """tiles: [n_tiles, 3] int32 {sequence, first row, end row} of at most `tile_rows` rows.
        64-row tiles run the 16x16 register kernel; 128 / 256-row tiles the LDS-staged 32x32
        kernel (bf16 KV cache, head dim 128: `prefill_tile_rows` says which the engine builds)."""
        T, n_q, hd = q.shape
        L, NB, n_kv, BS, _ = k_cache.shape
        _req(tiles is not None and tiles.dtype == torch.int32 and tiles.dim() == 2 and tiles.shape[1] == 3,
             "prefill attention needs the [n_tiles,3] int32 tile table")
        _req(q.is_contiguous() and block_tables.dtype == torch.int32 and q_start.dtype == torch.int32
             and seq_lens.dtype == torch.int32, "prefill attention inputs")
        out = torch.empty(T, n_q * hd, dtype=q.dtype, device=q.device)
        if tile_rows != 64:
            _req(tile_rows in (128, 256) and hd == 128 and not _kv_fp8(k_cache, v_cache),
                 "32x32 prefill attention: 128 / 256-row tiles, head dim 128, bf16 KV cache")
            _check(lib.bcg_paged_attention_prefill32(
                _p(q), _p(k_cache), _p(v_cache), layer, NB, n_kv, _p(block_tables), block_tables.shape[1],
                _p(q_start), _p(seq_lens), _p(tiles), tiles.shape[0], n_q, hd, BS, scale, _p(out),
                tile_rows, 0, _stream()), "paged_attention_prefill32")
            return out
        _check(lib.bcg_paged_attention_prefill(
            _p(q), _p(k_cache), _p(v_cache), layer, NB, n_kv, _p(block_tables), block_tables.shape[1],
            _p(q_start), _p(seq_lens), _p(tiles), tiles.shape[0], n_q, hd, BS, scale, _p(out),
            4, _kv_fp8(k_cache, v_cache), _stream()), "paged_attention_prefill")
        return out

    def prefill_tile_rows(hd, kv_fp8=False, max_blocks=0):
        """Rows per prefill attention tile for this geometry (the tile table the caller builds):
        128 / 256 select the LDS-staged 32x32 kernel (head dim 128, bf16 KV, block tables of at
        most 1024 entries -- 16k tokens -- which it stages in LDS), 64 the 16x16 one.
        BCG_PREFILL_TILE_ROWS overrides the default."""
        rows = int(os.environ.get("BCG_PREFILL_TILE_ROWS", PREFILL_TILE_ROWS))
        ok = rows in (128, 256) and hd == 128 and not kv_fp8 and max_blocks <= PREFILL32_MAX_BLOCKS
        return rows if ok else 64

    # Per-call GEMM dispatch log (which projection shapes reach a hand kernel, also
    # inside TP worker processes that no profiler sees): (M, N, K, epi, dtype) -> choice -> calls.
    # Off unless enabled (BCG_GEMM_LOG=1 or dispatch_log.enable()); graph-captured calls are
    # logged once, at capture (the replays run the same kernels).
    dispatch_log = SimpleNamespace(enabled=os.environ.get("BCG_GEMM_LOG") == "1", calls={})

    def _log(M, N, K, epi, choice, dtype="bf16"):
        if dispatch_log.enabled:
            key = (M, N, K, epi, dtype, "lib" if choice is None else f"{choice[0]}x{choice[1]}")
            dispatch_log.calls[key] = dispatch_log.calls.get(key, 0) + 1

    def _plain(x, w):
        """Operands that the kernels of this file take as they lie: bf16 on the current GPU, rows contiguous, 16-byte aligned, bare
        and not watched (the library's products carry gradients, tangents and transforms, these do not)."""
        return (x.dtype == w.dtype == torch.bfloat16 and x.is_cuda and x.device == w.device
                and x.get_device() == torch.cuda.current_device() and w.dim() == 2 and w.shape[1] == x.shape[1] and x.is_contiguous()
                and w.is_contiguous() and not watched() and bare(x) and bare(w) and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)

    def _plain_beside(t, shape, x):
        """The same for a bias, residual or norm weight beside x."""
        return (t.dtype == torch.bfloat16 and t.device == x.device and t.shape == shape and t.is_contiguous() and bare(t)
                and t.data_ptr() % 16 == 0)

    def _plain_bias(bias, N, x):
        return bias is None or _plain_beside(bias, (N,), x)

    def _mid(x, w, epi):
        """The plan by which the kernel for tens to hundreds of rows takes x W^T (csrc/kernels/gemm_mid.hip says which it does), else
        None (`few_rows_stay`)."""
        M, K = x.shape
        N = w.shape[0]
        if not (33 <= M <= MID_ROWS and plan.mode == "1") or (M <= SKINNY_ROWS and few_rows_stay(M, N, K, epi == 1) and few_rows_pay(M, N, 2 * K, epi == 1)):
            return None
        p = plan.mid(M, N, K, epi)
        return p if p is not None and _plain(x, w) else None

    def _gemm_mid(p, x, w, epi, out, bias=None, residual=None, scales=(None, None), N=None, at=0):
        """N, at: gated, N / 2 of the features from at / 2 on, into their columns of `out`."""
        M, K = x.shape
        inter = w.shape[0] // 2
        N = w.shape[0] if N is None else N
        ws = cnt = None
        if p >> 8 > 1:
            tiles = c_int()
            ws = torch.empty(lib.bcg_gemm_mid_parts(p, epi, M, N, ctypes.byref(tiles)), dtype=torch.float32, device=x.device)
            cnt = _counters(x.device)   # (at most 256 tiles: one round)
        _check(lib.bcg_gemm_mid(p, epi, _p(x), w.data_ptr() + at * K, *(None if t is None else _p(t) for t in (*scales, bias, residual)),
                                out.data_ptr() + at, None if ws is None else _p(ws), None if cnt is None else _p(cnt), M, N, K, inter,
                                _stream()), "gemm_mid")   # (at / 2 rows or features of 2 bytes)
        return out

    def _gemm_mid_act(p, x, w, out, other, at=0, tokens=None, off=0):
        """bcg_gemm_mid_act: at > 0, `other` takes the columns from `at` on through gelu; else gelu times columns off .. of the rows `tokens` of
        the table `other`."""
        M, K = x.shape
        N = w.shape[0]
        _log(M, N, K, 0, (MID_CFG, p))
        ws = cnt = None
        if p >> 8 > 1:
            tiles = c_int()
            ws = torch.empty(lib.bcg_gemm_mid_parts(p, 0, M, N, ctypes.byref(tiles)), dtype=torch.float32, device=x.device)
            cnt = _counters(x.device)
        _check(lib.bcg_gemm_mid_act(p, _p(x), _p(w), _p(out), other.data_ptr() + 2 * off, None if tokens is None else _p(tokens),
                                    None if ws is None else _p(ws), None if cnt is None else _p(cnt), M, N, K, at,
                                    0 if at else other.shape[1], 0 if at else other.shape[0], _stream()), "gemm_mid_act")

    def _pieces(x, w, epi, beside=None, shape=None):
        """Runs of rows and their choices (`GemmPlan.pieces`); beside: the bias or residual, of this shape.  Fewer rows than LARGE_M are
        one run whatever the operands are, so nothing is looked at there: a small eager step is bound by the host (24 layers of
        width 896, 456 rows: 4408 us with the look, 3810 without)."""
        M, K = x.shape
        if M < LARGE_M or not (_plain(x, w) and (beside is None or _plain_beside(beside, shape, x))):
            return [(M, plan.choose(M, w.shape[0], K, epi))]
        return plan.pieces(M, w.shape[0], K, epi)

    def _skinny(x, w, epi):
        """Whether the few-row kernel takes x W^T: up to SKINNY_ROWS rows of whole 128-byte lines, where they pay (csrc/kernels/
        gemm_skinny.hip holds more of both sides' times); table and library keep the others."""
        M, K = x.shape
        N = w.shape[0]
        return (plan.mode == "1" and 1 <= M <= SKINNY_ROWS and K % 64 == 0 and 64 <= K <= SKINNY_ROW_BYTES // 2
                and N >= 8 and N % (8 if epi == 1 else 4) == 0 and few_rows_pay(M, N, 2 * K, epi == 1) and _plain(x, w))

    def _skinny_name(M, K):
        """("skinny", blocks of 16 rows) in the dispatch log."""
        return ("skinny" if K <= SKINNY_LONG_K else "skinny_long", -(-M // 16))

    def _gemm_skinny(x, w, epi=0, bias=None, residual=None, norm_w=None, eps=0.0):
        M, K = x.shape
        N = w.shape[0]
        _log(M, N, K, epi, _skinny_name(M, K))
        out = residual if epi == 2 else torch.empty(M, N // 2 if epi == 1 else N, dtype=x.dtype, device=x.device)
        _check(lib.bcg_gemm_skinny(epi, _p(x), _p(w), None if norm_w is None else _p(norm_w), eps,
                                   None if bias is None else _p(bias), None if residual is None else _p(residual), _p(out),
                                   M, N, K, _stream()), "gemm_skinny")
        return out

    def linear(x, w, bias=None, _epi_log=0):
        """y = x W^T (+b): the few-row kernel, the hand MFMA GEMM where the plan says it beats hipBLASLt, hipBLASLt
        otherwise."""
        M, K = x.shape
        N = w.shape[0]
        p = _mid(x, w, 0)
        if p is not None and _plain_bias(bias, N, x):
            _log(M, N, K, _epi_log, (MID_CFG, p))
            return _gemm_mid(p, x, w, 0, torch.empty(M, N, dtype=x.dtype, device=x.device), bias)
        if _skinny(x, w, 0) and _plain_bias(bias, N, x):
            return _gemm_skinny(x, w, 0, bias)
        if not (x.is_contiguous() and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16):
            _log(M, N, K, _epi_log, None)
            return torch.nn.functional.linear(x, w, bias)
        parts = _pieces(x, w, 0, bias, (N,))
        if len(parts) == 1:
            return _linear_rows(x, w, bias, parts[0][1], None, _epi_log)
        out, at = torch.empty(M, N, dtype=x.dtype, device=x.device), 0
        for rows, cfg in parts:
            _linear_rows(x[at:at + rows], w, bias, cfg, out[at:at + rows], _epi_log)
            at += rows
        return out

    def _linear_rows(x, w, bias, cfg, out, epi_log):
        _log(x.shape[0], w.shape[0], x.shape[1], epi_log, cfg)
        if cfg is not None:
            return _hand(x, w, cfg, 0, out, bias=bias)
        if out is None:
            return torch.nn.functional.linear(x, w, bias)
        return torch.mm(x, w.t(), out=out) if bias is None else torch.addmm(bias, x, w.t(), out=out)

    from .gemm_plan import LARGE_M, MID_CFG, PP_CFG, SMALL_CFG, W4_CFG, GemmPlan
    plan = GemmPlan(lib)

    # Split-K arrival counters (one int per output tile; the last-arriving workgroup of a
    # tile resets its counter, so a buffer stays zero between launches).  Kernels that may
    # run CONCURRENTLY need disjoint buffers: every stream has its own for what is launched on it, and every
    # capture its own for what it records, as the graph may be replayed on any stream, beside others that were captured on the same one.
    counters = {}          # (device index, stream handle) -> int32 [65536]
    capture_counters = {}  # (device index, stream handle) -> (capture, int32 [65536]) of the last capture on that stream

    def _new_counters(dev):
        _req(not torch.cuda.is_current_stream_capturing(),
             "split-K counters must be allocated outside graph capture (ops.prepare_device)")
        return torch.zeros(1 << 16, dtype=torch.int32, device=dev)

    sk_ws = {}  # device index -> fp32 [2 x CUs x 65536]: stream-K parts (W4, split_k == 0)

    def prepare_device(dev):
        dev = torch.device(dev)
        if dev.index is None:
            dev = torch.device("cuda", torch.cuda.current_device())
        register_stream(torch.cuda.default_stream(dev))
        if dev.index not in sk_ws:  # (128 MiB; allocated outside any graph capture)
            with torch.cuda.device(dev):
                sk_ws[dev.index] = torch.empty(lib.bcg_gemm_w4_sk_ws_floats(), dtype=torch.float32, device=dev)

    def _sk_workspace(dev):
        dev = torch.device("cuda", dev.index if dev.index is not None else torch.cuda.current_device())
        if dev.index not in sk_ws:
            _req(not torch.cuda.is_current_stream_capturing(), "stream-K parts must be allocated outside graph capture (ops.prepare_device)")
            prepare_device(dev)
        return sk_ws[dev.index]

    def register_stream(stream):
        """Make `stream`'s split-K counters now, not at its first product."""
        key = (stream.device.index, stream.cuda_stream)
        if key not in counters:
            with torch.cuda.stream(stream):   # (zeroed there: its products are behind it)
                counters.setdefault(key, _new_counters(stream.device))

    def _counters(dev):
        """The current stream's counters, made at its first product; past 64 streams (the pool has 32) zeros for this product alone."""
        dev = torch.device("cuda", dev.index if dev.index is not None else torch.cuda.current_device())
        stream = torch.cuda.current_stream(dev)
        key = (dev.index, stream.cuda_stream)
        if torch.cuda.is_current_stream_capturing():
            return _capture_counters(dev, key)
        if key not in counters:
            if len(counters) >= 64:
                return _new_counters(dev)
            register_stream(stream)
        return counters[key]

    def _capture_counters(dev, key):
        """Out of the graph's own memory, zeroed where its first product on this stream is: every replay zeroes them before it uses them, and nobody
        else does.  Held while the capture lasts (after that it is the graph's: no product of another one is given them), until the
        next on the stream."""
        capture = lib.bcg_capture_id(key[1])
        held = capture_counters.get(key)
        if held is None or held[0] != capture or capture == 0:
            held = (capture, torch.zeros(1 << 16, dtype=torch.int32, device=dev))
            if capture != 0 and (key in capture_counters or len(capture_counters) < 64):
                capture_counters[key] = held
        return held[1]

    def gemm_nt(x, w, cfg, epi=0, bias=None, residual=None, out=None, split_k=1):
        """Hand MFMA GEMM (csrc/kernels/gemm.hip): x [M,K] @ w[N,K]^T with epilogue `epi`
        (0 store(+bias), 1 silu(gate)*up -> [M, N/2], 2 residual + acc); `split_k` K-slices
        reduced in the kernel by the last-arriving workgroup of each tile."""
        if isinstance(cfg, (tuple, list)):
            cfg, split_k = cfg
        M, K = x.shape
        N = w.shape[0]
        _req(x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.is_contiguous() and w.is_contiguous()
             and w.shape[1] == K, "gemm_nt: contiguous bf16 x [M,K], w [N,K]")
        _req(plan.supported(cfg, M, N, K, epi, split_k),
             f"gemm_nt: shape {M}x{N}x{K} epi {epi} split {split_k} unsupported by tile {cfg}")
        width = N // 2 if epi == 1 else N
        if out is None:
            out = torch.empty(M, width, dtype=x.dtype, device=x.device)
        _req(out.shape == (M, width) and out.is_contiguous() and out.dtype == torch.bfloat16, "gemm_nt: out")
        if bias is not None:
            _req(bias.shape == (N,) and bias.dtype == torch.bfloat16 and bias.is_contiguous(), "gemm_nt: bias")
        if epi == 2:
            _req(residual is not None and residual.shape == (M, N) and residual.is_contiguous()
                 and residual.dtype == torch.bfloat16, "gemm_nt: residual [M,N] bf16")
        ws = cnt = None
        if split_k == 0:  # W4 stream-K: the device's persistent part buffer + the counters
            ws, cnt = _sk_workspace(x.device), _counters(x.device)
        elif split_k > 1:
            bm, bn = plan.tiles[cfg]
            tiles = (M + bm - 1) // bm * ((N + bn - 1) // bn)
            _req(tiles <= (1 << 16), "gemm_nt: too many output tiles for split-K")
            ws = torch.empty(tiles * split_k * bm * bn, dtype=torch.float32, device=x.device)
            cnt = _counters(x.device)
        _check(lib.bcg_gemm_nt(cfg, epi, _p(x), _p(w), _p(bias) if bias is not None else None,
                               _p(residual) if residual is not None else None, _p(out),
                               _p(ws) if ws is not None else None, _p(cnt) if cnt is not None else None,
                               M, N, K, N // 2, split_k, _stream()), "gemm_nt")
        return out

    def _hand(x, w, cfg, epi, out, **beside):
        """A piece of a product (`_pieces`) by its choice.  The one-round kernel is chosen only where `_pieces` looked at the operands
        and comes with an `out` of its rows; `gemm_nt`, which anyone may call, refuses it like every configuration that it does not hold."""
        if cfg[0] == MID_CFG:
            return _gemm_mid(cfg[1], x, w, epi, out, **beside)
        return gemm_nt(x, w, cfg, epi, out=out, **beside)

    def linear_silu(x, w):
        """silu(x Wg^T) * (x Wu^T), W = [gate; up] -- K-ACT fused into the gate_up GEMM."""
        M, K = x.shape
        p = _mid(x, w, 1)
        if p is not None:
            _log(M, w.shape[0], K, 1, (MID_CFG, p))
            return _gemm_mid(p, x, w, 1, torch.empty(M, w.shape[0] // 2, dtype=x.dtype, device=x.device))
        if _skinny(x, w, 1):
            return _gemm_skinny(x, w, 1)
        if not (x.is_contiguous() and x.dtype == torch.bfloat16):
            return silu_mul(linear(x, w, _epi_log=1))
        N = w.shape[0]
        n1 = plan.columns(M, N, K)
        if n1 < N and _plain(x, w):
            out = torch.empty(M, N // 2, dtype=x.dtype, device=x.device)
            p = plan.mid(M, N - n1, K, 1)
            for cfg, at, n in ((W4_CFG, 0, n1), ((MID_CFG, p) if p is not None else SMALL_CFG, n1, N - n1)):   # both halves of w from row at / 2 on
                _log(M, n, K, 1, cfg if isinstance(cfg, tuple) else (cfg, 1))
                if isinstance(cfg, tuple):
                    _gemm_mid(p, x, w, 1, out, N=n, at=at)
                    continue
                _check(lib.bcg_gemm_nt(cfg, 1, _p(x), w.data_ptr() + at * K, None, None, out.data_ptr() + at, None, None, M, n, K, N // 2,
                                       1, _stream()), "gemm_nt")   # (at / 2 rows or features of 2 bytes)
            return out
        parts = _pieces(x, w, 1)
        if len(parts) == 1 and parts[0][1] is None:
            return silu_mul(linear(x, w, _epi_log=1))
        out, at = torch.empty(M, N // 2, dtype=x.dtype, device=x.device), 0
        for rows, cfg in parts:
            xr, dst = x[at:at + rows], out[at:at + rows]
            at += rows
            if cfg is None:
                dst.copy_(silu_mul(linear(xr, w, _epi_log=1)))
            else:
                _log(rows, N, K, 1, cfg)
                _hand(xr, w, cfg, 1, dst)
        return out

    def _w4_act(epi, x, w, c, tail, inter, limit):
        M, K = x.shape
        _log(M, w.shape[0], K, epi, (W4_CFG, 1))
        _check(lib.bcg_gemm_w4_act(epi, _p(x), _p(w), _p(c), None if tail is None else _p(tail), M, w.shape[0], K, inter, limit, _stream()),
               "gemm_w4_act")

    def linear_clamped_glu(x, w, limit):
        """gated_act(linear(x, w), "clamped_glu", limit), W = [gate; up]: one launch where `GemmPlan.clamped_tiles` says so."""
        M, K = x.shape
        if not (limit > 0 and plan.clamped_tiles(M, w.shape[0], K) and _plain(x, w)):
            return extra["gated_act"](linear(x, w), "clamped_glu", limit)
        out = torch.empty(M, w.shape[0] // 2, dtype=x.dtype, device=x.device)
        _w4_act(5, x, w, out, None, w.shape[0] // 2, float(limit))
        return out

    def linear_tail_gelu(x, w, at):
        """(y, hidden): y = linear(x, w) and None, or, where one launch takes the activation along (`GemmPlan.tail_tiles`, the kernel for
        tens to hundreds of rows), the first `at` columns of it and act_fn of the others, "gelu_tanh"."""
        M, K = x.shape
        N = w.shape[0]
        tiles = plan.tail_tiles(M, N, K, at)
        p = None if tiles or not (0 < at < N and at % 8 == 0) else _mid(x, w, 0)
        if p is None and not (tiles and _plain(x, w)):
            return linear(x, w), None
        y = torch.empty(M, at, dtype=x.dtype, device=x.device)
        hidden = torch.empty(M, N - at, dtype=x.dtype, device=x.device)
        if p is not None:
            _gemm_mid_act(p, x, w, y, hidden, at=at)
        else:
            _w4_act(6, x, w, y, hidden, at, 0.0)
        return y, hidden

    def linear_gelu_table(x, w, tokens, table, off):
        """gelu_gather_mul(linear(x, w), tokens, table, off), in one launch where the kernel for tens to hundreds of rows takes the product."""
        N = w.shape[0]
        p = _mid(x, w, 0)
        if p is None or not (table.dim() == 2 and table.dtype == x.dtype and table.device == x.device and table.is_contiguous() and bare(table)
                             and table.shape[1] % 8 == 0 and off % 8 == 0 and 0 <= off <= table.shape[1] - N and table.data_ptr() % 16 == 0
                             and tokens.dtype == torch.int32 and tokens.is_contiguous() and tokens.device == x.device
                             and tokens.numel() == x.shape[0]):
            return extra["gelu_gather_mul"](linear(x, w), tokens, table, off)
        out = torch.empty(x.shape[0], N, dtype=x.dtype, device=x.device)
        _gemm_mid_act(p, x, w, out, table, tokens=tokens, off=off)
        return out

    def _norm_fusable(x, w_norm):
        return x.shape[0] <= SKINNY_NORM_ROWS and x.shape[1] <= 8192 and _plain_beside(w_norm, (x.shape[1],), x)

    def norm_linear(x, w_norm, eps, w, bias=None):
        """linear(rmsnorm(x, w_norm, eps), w, bias), one kernel for a few rows."""
        if x.dim() == 2 and _skinny(x, w, 0) and _norm_fusable(x, w_norm) and _plain_bias(bias, w.shape[0], x):
            return _gemm_skinny(x, w, 0, bias, norm_w=w_norm, eps=eps)
        return linear(rmsnorm(x, w_norm, eps), w, bias)

    def norm_linear_silu(x, w_norm, eps, w):
        """linear_silu(rmsnorm(x, w_norm, eps), w), one kernel for a few rows."""
        if x.dim() == 2 and _skinny(x, w, 1) and _norm_fusable(x, w_norm):
            return _gemm_skinny(x, w, 1, norm_w=w_norm, eps=eps)
        return linear_silu(rmsnorm(x, w_norm, eps), w)

    residual_addmm = os.environ.get("BCG_RESIDUAL_ADDMM", "1") == "1"

    def linear_residual(x, w, residual):
        """residual <- residual + x W^T (in place; the o/down projection fused with the
        residual-stream update of the next add+RMSNorm).  Returns `residual`."""
        M, K = x.shape
        p = _mid(x, w, 2)
        if p is not None and _plain_beside(residual, (M, w.shape[0]), x):
            _log(M, w.shape[0], K, 2, (MID_CFG, p))
            return _gemm_mid(p, x, w, 2, residual, residual=residual)
        if _skinny(x, w, 2) and _plain_beside(residual, (M, w.shape[0]), x):
            return _gemm_skinny(x, w, 2, residual=residual)
        parts = [(M, None)]
        if x.is_contiguous() and x.dtype == torch.bfloat16:
            parts = _pieces(x, w, 2, residual, (M, w.shape[0]))
        at = 0
        for rows, cfg in parts:
            whole = rows == M
            _residual_rows(x if whole else x[at:at + rows], w, residual if whole else residual[at:at + rows], cfg)
            at += rows
        return residual

    def _residual_rows(x, w, residual, cfg):
        M, K = x.shape
        _log(M, w.shape[0], K, 2, cfg)
        if cfg is not None:
            _hand(x, w, cfg, 2, residual, residual=residual)
        elif (residual_addmm and residual.is_contiguous() and residual.dtype == x.dtype == w.dtype
                and residual.shape == (M, w.shape[0])):
            # hipBLASLt with beta = 1: the residual add rides in the GEMM epilogue (one read
            # of the residual, no separate elementwise pass over three [M, H] tensors)
            residual.addmm_(x, w.t())
        else:
            residual.add_(torch.nn.functional.linear(x, w))

    def sample_step(logits, fsm_next, fsm_dist, fsm_base, fsm_state, gen_count, max_new, temperature,
                    row_keys, done, seq_lens, out_tokens, next_tokens, seed, budget_aware, n_text_tokens,
                    eos_id, eos_id2):
        B, V = logits.shape
        _req(logits.dtype == torch.bfloat16 and logits.is_contiguous(), "logits bf16 [B,V]")
        _req(fsm_next.dtype == torch.int16 and fsm_next.shape[1] == V and fsm_dist.dtype == torch.int16,
             "fsm tables int16 [rows,V]")
        for t in (fsm_base, fsm_state, gen_count, max_new, row_keys, done, seq_lens, next_tokens):
            _req(t.dtype == torch.int32 and t.numel() == B and t.is_contiguous(), "per-row int32 state")
        _req(temperature.dtype == torch.float32 and out_tokens.dtype == torch.int32
             and out_tokens.shape[0] == B, "temperature/out_tokens")
        _check(lib.bcg_guided_sample(
            _p(logits), B, V, _p(fsm_next), _p(fsm_dist), _p(fsm_base), _p(fsm_state), _p(gen_count),
            _p(max_new), _p(temperature), _p(row_keys), _p(done), _p(seq_lens), _p(out_tokens),
            out_tokens.shape[1], _p(next_tokens), seed & 0xFFFFFFFF, int(bool(budget_aware)), n_text_tokens,
            eos_id, eos_id2, _stream()), "guided_sample")

    f8 = torch.float8_e4m3fn

    def quant_fp8(x):
        _req(x.dtype == torch.bfloat16 and x.is_contiguous() and x.dim() == 2 and x.shape[1] % 8 == 0,
             "quant_fp8: bf16 [T,K], K % 8 == 0")
        T, K = x.shape
        q = torch.empty(T, K, dtype=f8, device=x.device)
        s = torch.empty(T, dtype=torch.float32, device=x.device)
        _check(lib.bcg_quant_fp8(_p(x), _p(q), _p(s), T, K, _stream()), "quant_fp8")
        return q, s

    def add_rmsnorm_fp8(x, residual, w, eps):
        _req(x.dtype == torch.bfloat16 and x.is_contiguous() and x.dim() == 2, "add_rmsnorm_fp8: x bf16 [T,H]")
        T, H = x.shape
        _req(w.shape == (H,) and w.dtype == torch.bfloat16, "add_rmsnorm_fp8: weight [H] bf16")
        has_res = residual is not None
        if not has_res:
            residual = torch.empty_like(x)
        else:
            _req(residual.shape == x.shape and residual.is_contiguous(), "add_rmsnorm_fp8: residual shape")
        q = torch.empty(T, H, dtype=f8, device=x.device)
        s = torch.empty(T, dtype=torch.float32, device=x.device)
        _check(lib.bcg_add_rmsnorm_fp8(_p(x), _p(residual), _p(w), _p(q), _p(s), T, H, eps, int(has_res),
                                       _stream()), "add_rmsnorm_fp8")
        return q, s, residual

    def rmsnorm_fp8(x, w, eps):
        """Plain RMSNorm + row-wise fp8 quant (the residual stream was updated by the GEMM epilogue)."""
        _req(x.dtype == torch.bfloat16 and x.is_contiguous() and x.dim() == 2, "rmsnorm_fp8: x bf16 [T,H]")
        T, H = x.shape
        _req(w.shape == (H,) and w.dtype == torch.bfloat16, "rmsnorm_fp8: weight [H] bf16")
        q = torch.empty(T, H, dtype=f8, device=x.device)
        s = torch.empty(T, dtype=torch.float32, device=x.device)
        _check(lib.bcg_add_rmsnorm_fp8(_p(x), None, _p(w), _p(q), _p(s), T, H, eps, 2, _stream()), "rmsnorm_fp8")
        return q, s

    def embed_rmsnorm_fp8(tokens, table, w, eps):
        """(fp8(rmsnorm(table[tokens]) * w), row scales, table[tokens]) in one pass."""
        _req(tokens.dtype == torch.int32 and tokens.is_contiguous() and tokens.dim() == 1, "tokens int32 [T]")
        _req(table.dtype == torch.bfloat16 and table.is_contiguous() and table.dim() == 2, "table bf16 [V,H]")
        T, H = tokens.numel(), table.shape[1]
        _req(w.shape == (H,) and w.dtype == torch.bfloat16, "embed_rmsnorm_fp8: weight [H] bf16")
        residual = torch.empty(T, H, dtype=table.dtype, device=table.device)
        q = torch.empty(T, H, dtype=f8, device=table.device)
        s = torch.empty(T, dtype=torch.float32, device=table.device)
        _check(lib.bcg_embed_rmsnorm_fp8(_p(tokens), _p(table), _p(w), _p(residual), _p(q), _p(s), T, H, eps,
                                         _stream()), "embed_rmsnorm_fp8")
        return q, s, residual

    def silu_mul_fp8(gu):
        _req(gu.dtype == torch.bfloat16 and gu.is_contiguous() and gu.dim() == 2 and gu.shape[1] % 16 == 0,
             "silu_mul_fp8: bf16 [T,2I]")
        T, I2 = gu.shape
        q = torch.empty(T, I2 // 2, dtype=f8, device=gu.device)
        s = torch.empty(T, dtype=torch.float32, device=gu.device)
        _check(lib.bcg_silu_mul_fp8(_p(gu), _p(q), _p(s), T, I2 // 2, _stream()), "silu_mul_fp8")
        return q, s

    def gemm_nt_fp8(xq, xs, wq, ws, cfg, epi=0, bias=None, residual=None, out=None, split_k=1):
        """Hand fp8 MFMA GEMM (csrc/kernels/gemm.hip, F8): xs[m] * ws[n] * (xq . wq^T)
        (+ bias) (+ residual when epi == 2), e4m3fn operands, bf16 out."""
        if isinstance(cfg, (tuple, list)):
            cfg, split_k = cfg
        M, K = xq.shape
        N = wq.shape[0]
        _req(xq.dtype == f8 and wq.dtype == f8 and xq.is_contiguous() and wq.is_contiguous() and wq.shape[1] == K,
             "gemm_nt_fp8: contiguous e4m3fn xq [M,K], wq [N,K]")
        _req(xs.dtype == torch.float32 and xs.numel() == M and xs.is_contiguous() and ws.dtype == torch.float32
             and ws.numel() == N and ws.is_contiguous(), "gemm_nt_fp8: fp32 scales xs [M], ws [N]")
        bm, bn = plan.tiles[cfg]
        pp = cfg == PP_CFG  # 256 x 256 ping-pong kernel: N only a multiple of 16, 32-bit buffer offsets
        w4 = cfg == W4_CFG  # four-wave 256 x 256 kernel: N a multiple of 16, offsets below 2 GiB
        _req(0 <= cfg <= W4_CFG and K % 128 == 0 and N % (16 if pp or w4 else bn) == 0 and 1 <= split_k <= K // 128
             and epi in (0, 2) and (not pp or (M * K < 1 << 32 and N * K < 1 << 32))
             and (not w4 or ((M + 256) * K < 1 << 31 and (N + 256) * K < 1 << 31))
             and (not (pp or w4) or 2 * (M + 256) * N < 1 << 31),
             f"gemm_nt_fp8: shape {M}x{N}x{K} epi {epi} split {split_k} unsupported by tile {cfg}")
        if out is None:
            out = torch.empty(M, N, dtype=torch.bfloat16, device=xq.device)
        _req(out.shape == (M, N) and out.is_contiguous() and out.dtype == torch.bfloat16, "gemm_nt_fp8: out")
        if bias is not None:
            _req(bias.shape == (N,) and bias.dtype == torch.bfloat16 and bias.is_contiguous(), "gemm_nt_fp8: bias")
        if epi == 2:
            _req(residual is not None and residual.shape == (M, N) and residual.is_contiguous()
                 and residual.dtype == torch.bfloat16, "gemm_nt_fp8: residual [M,N] bf16")
        wsp = cnt = None
        if split_k > 1:
            tiles = (M + bm - 1) // bm * ((N + bn - 1) // bn)
            _req(tiles <= (1 << 16), "gemm_nt_fp8: too many output tiles for split-K")
            wsp = torch.empty(tiles * split_k * bm * bn, dtype=torch.float32, device=xq.device)
            cnt = _counters(xq.device)
        _check(lib.bcg_gemm_nt_fp8(cfg, epi, _p(xq), _p(wq), _p(xs), _p(ws), _p(bias) if bias is not None else None,
                                   _p(residual) if residual is not None else None, _p(out),
                                   _p(wsp) if wsp is not None else None, _p(cnt) if cnt is not None else None,
                                   M, N, K, split_k, _stream()), "gemm_nt_fp8")
        return out

    from .gemm_plan import Fp8Plan
    fp8_plan = Fp8Plan(plan.tiles)
    fp8_cfg = fp8_plan.choose

    def _skinny_fp8(xq, xs, wq, ws, *beside):
        """Whether the few-row kernel takes the fp8 product: as `_skinny`, every size up to 16 rows, past them rows of up to 8192 bytes and
        many longer ones (N, K of 256 to 16384, 1 to 32 rows, against tile kernels and library: 0.33 to 1.0); `beside`: [(bias or
        residual, its shape)]."""
        M, K = xq.shape
        N = wq.shape[0]
        return (plan.mode == "1" and 1 <= M <= 32 and K % 128 == 0 and 128 <= K <= SKINNY_ROW_BYTES and N >= 16 and N % 16 == 0
                and (M <= 16 or K <= 8192 or N >= 4096) and _plain_fp8(xq, xs, wq, ws, beside))

    def _plain_fp8(xq, xs, wq, ws, beside):
        """`_plain` for the fp8 products: operands, their scales and what stands beside them."""
        return (wq.dim() == 2 and wq.shape[1] == xq.shape[1]
                and xq.is_cuda and xq.get_device() == torch.cuda.current_device() and xq.is_contiguous() and wq.is_contiguous()
                and all(t.device == xq.device and t.data_ptr() % 16 == 0 and bare(t) for t in (xq, wq, xs, ws))
                and xs.dtype == ws.dtype == torch.float32 and xs.numel() == xq.shape[0] and ws.numel() == wq.shape[0] and xs.is_contiguous()
                and ws.is_contiguous() and not watched()
                and all(t is None or _plain_beside(t, shape, xq) for t, shape in beside))

    def _mid_fp8(xq, xs, wq, ws, *beside):
        """`_mid` for the fp8 products."""
        M, K = xq.shape
        if not (33 <= M <= MID_ROWS and plan.mode == "1"):
            return None
        p = lib.bcg_gemm_mid_plan(0, M, wq.shape[0], K, 1)
        return p if p >= 0 and _plain_fp8(xq, xs, wq, ws, beside) else None

    def _gemm_skinny_fp8(xq, xs, wq, ws, epi=0, bias=None, residual=None):
        M, K = xq.shape
        N = wq.shape[0]
        _log(M, N, K, epi, _skinny_name(M, K), "fp8")
        out = residual if epi == 2 else torch.empty(M, N, dtype=torch.bfloat16, device=xq.device)
        _check(lib.bcg_gemm_skinny_fp8(epi, _p(xq), _p(wq), _p(xs), _p(ws), None if bias is None else _p(bias),
                                       None if residual is None else _p(residual), _p(out), M, N, K, _stream()), "gemm_skinny_fp8")
        return out

    def linear_fp8(xq, xs, wq, ws, bias=None, out_dtype=torch.bfloat16):
        """fp8 projection with row-wise activation and per-channel weight scales: the hand
        fp8 MFMA kernel for decode-sized M, hipBLASLt (torch._scaled_mm) otherwise."""
        _req(xq.dtype == f8 and wq.dtype == f8 and xq.shape[1] == wq.shape[1], "linear_fp8 operands")
        if out_dtype == torch.bfloat16 and _skinny_fp8(xq, xs, wq, ws, (bias, (wq.shape[0],))):
            return _gemm_skinny_fp8(xq, xs, wq, ws, 0, bias)
        p = _mid_fp8(xq, xs, wq, ws, (bias, (wq.shape[0],))) if out_dtype == torch.bfloat16 else None
        if p is not None:
            _log(xq.shape[0], wq.shape[0], xq.shape[1], 0, (MID_CFG, p), "fp8")
            return _gemm_mid(p, xq, wq, 0, torch.empty(xq.shape[0], wq.shape[0], dtype=torch.bfloat16, device=xq.device), bias, scales=(xs, ws))
        cfg = None
        if out_dtype == torch.bfloat16 and xq.is_contiguous() and wq.is_contiguous():
            cfg = fp8_cfg(xq.shape[0], wq.shape[0], xq.shape[1])
        _log(xq.shape[0], wq.shape[0], xq.shape[1], 0, cfg, "fp8")
        if cfg is not None:
            return gemm_nt_fp8(xq, xs.contiguous(), wq, ws.contiguous(), cfg, 0, bias=bias)
        return torch._scaled_mm(xq, wq.t(), scale_a=xs.view(-1, 1), scale_b=ws.view(1, -1), bias=bias,
                                out_dtype=out_dtype)

    def linear_fp8_residual(xq, xs, wq, ws, residual):
        """residual <- residual + dequant(xq . wq^T) in place: the o/down projection's residual
        update in the hand fp8 kernel's epilogue (hipBLASLt + a separate add otherwise)."""
        _req(residual.dtype == torch.bfloat16 and residual.is_contiguous()
             and residual.shape == (xq.shape[0], wq.shape[0]), "linear_fp8_residual: residual [M,N] bf16")
        if xq.dtype == wq.dtype == f8 and _skinny_fp8(xq, xs, wq, ws, (residual, residual.shape)):
            return _gemm_skinny_fp8(xq, xs, wq, ws, 2, residual=residual)
        p = _mid_fp8(xq, xs, wq, ws, (residual, residual.shape)) if xq.dtype == wq.dtype == f8 else None
        if p is not None:
            _log(xq.shape[0], wq.shape[0], xq.shape[1], 2, (MID_CFG, p), "fp8")
            return _gemm_mid(p, xq, wq, 2, residual, residual=residual, scales=(xs, ws))
        if xq.is_contiguous() and wq.is_contiguous():
            cfg = fp8_cfg(xq.shape[0], wq.shape[0], xq.shape[1])
            if cfg is not None:
                return gemm_nt_fp8(xq, xs.contiguous(), wq, ws.contiguous(), cfg, 2, residual=residual,
                                   out=residual)
        return residual.add_(linear_fp8(xq, xs, wq, ws))

    from .seqmix import seqmix_ops
    from .seqstate import seqstate_ops
    extra = seqmix_ops(lib, linear, _counters)
    extra.update(seqstate_ops(lib))
    from .seqlatent import seqlatent_ops
    extra.update(seqlatent_ops(lib, extra.pop("_experts")))
    from .seqhyper import seqhyper_ops
    extra.update(seqhyper_ops(lib))

    return SimpleNamespace(name="hip", **extra, rmsnorm_fp8=rmsnorm_fp8, embed_rmsnorm_fp8=embed_rmsnorm_fp8,
                           linear_fp8_residual=linear_fp8_residual, linear=linear, norm_linear=norm_linear, norm_linear_silu=norm_linear_silu, linear_silu=linear_silu, linear_residual=linear_residual,
                           linear_clamped_glu=linear_clamped_glu, linear_tail_gelu=linear_tail_gelu, linear_gelu_table=linear_gelu_table,
                           gemm_nt=gemm_nt, gemm_plan=plan, prepare_device=prepare_device,
                           register_stream=register_stream, quant_fp8=quant_fp8, add_rmsnorm_fp8=add_rmsnorm_fp8,
                           silu_mul_fp8=silu_mul_fp8, linear_fp8=linear_fp8, gemm_nt_fp8=gemm_nt_fp8, fp8_cfg=fp8_cfg, rmsnorm=rmsnorm, add_rmsnorm=add_rmsnorm, silu_mul=silu_mul,
                           embed_rmsnorm=embed_rmsnorm,
                           qk_norm_rope_kv_write=qk_norm_rope_kv_write,
                           paged_attention_decode=paged_attention_decode,
                           decode_attention_pairs=decode_attention_pairs, decode_order=decode_order,
                           decode_workspace_numel=decode_workspace_numel,
                           decode_max_context=lambda cascade=True: lib.bcg_decode_max_context(int(cascade)),
                           paged_attention_prefill=paged_attention_prefill,
                           prefill_tile_rows=prefill_tile_rows,
                           sample_step=sample_step, dispatch_log=dispatch_log,
                           library=lib)
