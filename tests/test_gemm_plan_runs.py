"""The rules that split a projection into runs of rows or columns (`GemmPlan.pieces`, `GemmPlan.columns`), over random
shapes without a GPU: every row and column is covered once, each run is one that its kernel supports, and
shapes that the general path takes alone still do."""
import random

import pytest
import torch

from byzantine_consensus_llm_agents_amd.ops.gemm_plan import CUS, LARGE_M, SMALL_CFG, W4_CFG, GemmPlan


def _shapes(n):
    rng = random.Random(3)
    for _ in range(n):
        yield (rng.choice([1, 16, 17, 255, 256, 257, 448, 512, 700, 1024, 2047, 2048, 2049, 4449, 8183, 16384, rng.randint(1, 20000)]),
               rng.choice([16, 64, 1792, 4096, 5056, 22528, 24576, 34816, 16 * rng.randint(1, 3000), 256 * rng.randint(1, 200), rng.randint(1, 40000)]),
               rng.choice([64, 896, 4096, 5120, 17408, 64 * rng.randint(1, 300), rng.randint(1, 9000)]), rng.choice([0, 1, 2]))


def test_runs_of_rows():
    plan = GemmPlan()
    plan.mode = "1"
    split = 0
    for M, N, K, epi in _shapes(20000):
        runs = plan.pieces(M, N, K, epi)
        assert sum(r for r, _ in runs) == M and len(runs) <= 2 and all(r > 0 for r, _ in runs)
        for r, c in runs:
            assert c is None or plan.supported(c[0], r, N, K, epi, c[1]), (M, N, K, epi, runs)
        if M < LARGE_M or (M, N, K, epi) in plan.table:
            assert runs == [(M, plan.choose(M, N, K, epi))]
        split += len(runs) > 1
    assert split


def test_columns():
    plan = GemmPlan()
    plan.mode = "1"
    split = 0
    for M, N, K, _ in _shapes(40000):
        n1 = plan.columns(M, N, K)
        assert 0 < n1 <= N
        if n1 < N:
            assert 256 < M < LARGE_M and n1 % 256 == 0 and N % 256 == 0
            assert plan.supported(W4_CFG, M, n1, K, 1) and plan.supported(SMALL_CFG, M, N - n1, K, 1)
            whole = n1 // 256 * -(-M // 256)
            assert whole >= 0.94 * CUS * -(-whole // CUS)
            split += 1
    assert split


LIB, LARGE = None, (W4_CFG, 1)


@pytest.mark.parametrize("M,N,K,epi,runs", [
    (4098, 4096, 896, 2, [(4096, LIB), 2]), (8201, 12288, 960, 0, [(8192, LIB), 9]),          # rounds exactly full
    (2820, 5632, 896, 0, [(2816, LIB), 4]), (2565, 12800, 896, 0, [(2560, LIB), 5]), (8706, 7680, 896, 2, [(8704, LIB), 2]),
    (8723, 5632, 896, 2, [(8704, LARGE), 19]), (5384, 15104, 960, 0, [(5376, LARGE), 8]),     # 3 and 5 rounds but for a few tiles
    (7172, 13568, 960, 0, [(7168, LARGE), 4]),                                                # 6
    (16098, 7168, 960, 0, [(16098, LIB)]), (7678, 6144, 960, 0, [(7678, LIB)]),               # no split: 7 and 3 even rounds
    (11612, 4096, 960, 0, [(11612, LARGE)]), (2478, 16384, 960, 0, [(2478, LARGE)]),          # 3 uneven ones
    (9010, 4608, 10304, 0, [(9010, LARGE)]), (9010, 4608, 10176, 0, [(9010, LIB)]),           # 3 even ones, either side of LONG_K
    (2318, 6784, 896, 0, [(2304, LARGE), 14]), (8195, 11792, 896, 0, [(8192, LARGE), 3]),     # N not a multiple of 256
    (2617, 10304, 512, 0, [(2617, LARGE)]), (7982, 8016, 512, 2, [(7982, LIB)]), (8796, 9232, 512, 0, [(8796, LIB)]),
    (7939, 9216, 512, 0, [(7939, LARGE)]), (8183, 11264, 512, 0, [(8183, LARGE)]), (3858, 12544, 512, 0, [(3858, LIB)]),
    (5409, 3072, 896, 1, [(5376, LARGE), 33]), (4462, 4096, 512, 1, [(4462, LARGE)]), (2300, 9728, 2048, 1, [(2300, LARGE)]),
    (2300, 9728, 2112, 1, [(2300, LIB)]), (2300, 8192, 2048, 1, [(2048, LARGE), 252]), (4365, 2048, 512, 1, [(4365, LIB)])])
def test_who_takes_the_rounds(M, N, K, epi, runs):
    plan = GemmPlan(table=None)
    plan.mode, plan.max_m = "1", 0      # (no table, no rule for small steps: the library unless a rule of `pieces` says otherwise)
    got = plan.pieces(M, N, K, epi)
    assert got == [r if isinstance(r, tuple) else (r, LIB) for r in runs]


@pytest.mark.parametrize("mode", ["0", "force"])
def test_other_modes_split_nothing(mode):
    plan = GemmPlan()
    plan.mode = mode
    for M, N, K, epi in _shapes(2000):
        assert plan.columns(M, N, K) == N and plan.pieces(M, N, K, epi) == [(M, plan.choose(M, N, K, epi))]


def test_gated_columns_of_a_weight_past_32_bits():
    """A few columns of a gated weight whose up rows lie past the 32-bit offsets are refused before any launch (no GPU)."""
    import ctypes
    import os
    from byzantine_consensus_llm_agents_amd.ops.hip import load_library
    from byzantine_consensus_llm_agents_amd.utils.build import kernels_target
    if not os.path.exists(kernels_target()):
        pytest.skip("kernel library not built")
    one = ctypes.c_void_p(16)
    for inter, K in ((1 << 20, 1024), (1 << 19, 2048), ((1 << 20) - 128, 1024), (-128, 64)):     # 2 (2 inter + 256) K bytes: 2^31 and more
        assert load_library().bcg_gemm_nt(W4_CFG, 1, one, one, None, None, one, None, None, 256, 256, K, inter, 1, None) == -2


@pytest.mark.skipif(torch.cuda.device_count() > 0, reason="calls the entry points with addresses of nothing: the launch has to fail")
def test_activation_rules_take_what_their_kernel_takes():
    """The rules of the activations in the 256 x 256 kernel's epilogue and the bounds of its entry point at 32-bit offsets: a size
    that a rule takes is never refused (-2) there, one past the bounds never taken."""
    import ctypes
    import os
    from byzantine_consensus_llm_agents_amd.ops.hip import load_library
    from byzantine_consensus_llm_agents_amd.utils.build import kernels_target
    if not os.path.exists(kernels_target()):
        pytest.skip("kernel library not built")
    lib, plan, one = load_library(), GemmPlan(), ctypes.c_void_p(16)
    taken = refused = 0
    for M in (512, 4096, 16384, 21589, 43700, 65536, 87126, 87125, 131072 - 256):
        for ff, K in ((8192, 2048), (12288, 2048), (12288, 4096), (32768, 4096), (65536, 1024), (131072, 2048), (524160, 1024)):
            for N, epi, at, rule in ((2 * ff, 5, ff, plan.clamped_tiles(M, 2 * ff, K)), (ff + 768, 6, 768, plan.tail_tiles(M, ff + 768, K, 768))):
                got = lib.bcg_gemm_w4_act(epi, one, one, one, one, M, N, K, at, 1.0, None)
                assert not (rule and got == -2), (M, N, K, epi)
                taken, refused = taken + rule, refused + (got == -2)
    assert plan.clamped_tiles(16384, 65536, 4096) and taken > 20 and refused > 20
