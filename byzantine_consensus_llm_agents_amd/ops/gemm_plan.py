"""Which GEMM runs where: the hand MFMA kernel (csrc/kernels/gemm.hip) or hipBLASLt.

Up to 64 rows the few-row kernel (csrc/kernels/gemm_skinny.hip) and 33 to 1536 rows the one-round kernel
(csrc/kernels/gemm_mid.hip, `GemmPlan.mid`) come before this choice where their own rules take a product.  What they
leave (decode buckets whose product is more than a round of tiles, operands they refuse) goes by a table per (M, N, K,
epilogue) measured on the GPU (``tools/tune_hand_gemm.py`` -> ``engine/tuned/hand_gemm.json``: for every decode bucket
and projection shape, every tile configuration and the library are timed and the fastest is kept), prefill chunks by
the rules of `GemmPlan.pieces`, and shapes that nothing covers stay on the library.
Most entries of 33 to 1536 rows serve only operands that the one-round kernel refuses (not contiguous, not on 16 bytes, watched by autograd).

``BCG_HAND_GEMM``: ``0`` = library only, ``1`` (default) = table / rule,
``force`` = hand kernel wherever the shape is supported (tests; ``BCG_HAND_GEMM_SPLIT``
= the split-K to force with it).

"""

import bisect
import ctypes
import json
import os
from typing import Dict, List, Optional, Tuple

TABLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "engine", "tuned",
                     "hand_gemm.json")
TILES = ((128, 128), (64, 128), (128, 64), (256, 128), (64, 256), (64, 64), (32, 128),  # csrc/kernels/gemm.hip CFGS
         (256, 128), (128, 256), (128, 128), (256, 256), (256, 256))
PP_CFG = 10  # csrc/kernels/gemm_pp.hip: 256 x 256 ping-pong tile, N only a multiple of 16
W4_CFG = 11  # csrc/kernels/gemm_w4.hip: 256 x 256, four 128 x 128 waves (one per SIMD), LDS-DMA fed
BIG_CFGS = (PP_CFG, W4_CFG)  # 256 x 256 tiles (the register-staged form lost its A/B: csrc/experimental/gemm_rs.hip)
SMALL_CFG = 5  # 64 x 64
MID_CFG = 12  # csrc/kernels/gemm_mid.hip: a tile of its own for every product, its plan in the place of the split
N_CFGS = len(TILES)
SPLITS = (1, 2, 3, 4, 6, 8)
CUS = 256       # compute units of an MI355X; on a part of one the rounds would be sized wrongly, the results the same
LARGE_M = 2048    # `pieces`: from here on the row count is a prefill step's
LONG_K = 10240    # from here on the library's rate follows the rounds less
W4_KTILE_US = 1.46   # one wave of 256 x 256 tiles: microseconds per 64 of K (512 tiles, K = 4096 .. 17408)
STREAM_K = 0  # split_k value of the W4 kernel's stream-K launch (one workgroup per CU over tiles x K-tiles)


class GemmPlan:
    def __init__(self, lib=None, table: Optional[str] = TABLE, max_m: int = 1024):
        self.mode = os.environ.get("BCG_HAND_GEMM", "1")
        self.lib = lib
        self.force_split = int(os.environ.get("BCG_HAND_GEMM_SPLIT", "1"))  # split-K in "force" mode (tests)
        self.max_m = max_m
        self.rows: Dict[Tuple[int, int, int], List[int]] = {}
        self.timings: Dict[Tuple[int, int, int, int], Dict[str, float]] = {}
        self.tiles = {}
        for cfg in range(N_CFGS):
            self.tiles[cfg] = TILES[cfg]
            if lib is not None:  # the library is the source of truth
                bm, bn = ctypes.c_int(), ctypes.c_int()
                if lib.bcg_gemm_tile(cfg, ctypes.byref(bm), ctypes.byref(bn)) == 0:
                    self.tiles[cfg] = (bm.value, bn.value)
        self.table: Dict[Tuple[int, int, int, int], Tuple[int, int]] = {}
        self.kept: Dict[Tuple[int, int, int, int], int] = {}   # entries that the one-round kernel does not beat: from which row count on
        if table and os.path.exists(table):
            with open(table) as fh:
                data = json.load(fh)
            for key, choice in data.get("choice", {}).items():
                m, n, k, e = map(int, key.split(","))
                self.table[(m, n, k, e)] = tuple(choice) if isinstance(choice, list) else (int(choice), 1)
            for (m, n, k, e) in sorted(self.table):     # measured row counts of every shape, in order
                self.rows.setdefault((n, k, e), []).append(m)
            self.kept = {tuple(map(int, key.split(","))): rows for key, rows in data.get("beats_one_round", {}).items()}
            for key, times in data.get("timings_us", {}).items():
                self.timings[tuple(map(int, key.split(",")))] = times

    def supported(self, cfg: int, M: int, N: int, K: int, epi: int, split_k: int = 1) -> bool:
        if split_k == STREAM_K:  # W4 only: an arrival counter per tile, 32-bit unit arithmetic
            tiles = -(-M // 256) * -(-N // 256)
            if cfg != W4_CFG or tiles > 65024 or tiles * (K // 64) * 256 >= 1 << 31:
                return False
            split_k = 1
        if cfg not in self.tiles or M <= 0 or K % 64 or K <= 0 or split_k < 1 or K // 64 < split_k:
            return False
        if cfg == W4_CFG and split_k > 1 and -(-M // 256) * -(-N // 256) > 65024:
            return False  # split-K arrival counters below the reduce-scatter scheme's slots
        bn = self.tiles[cfg][1]
        if cfg in BIG_CFGS:  # 32-bit buffer offsets: operands below 4 GiB (W4: 2 GiB), output below 2 GiB
            lim = 1 << (31 if cfg == W4_CFG else 32)
            ldc = N // 2 if epi == 1 else N
            return (N % 16 == 0 and 2 * (M + 256) * K < lim and 2 * (N + 256) * K < lim
                    and 2 * (M + 256) * ldc < 1 << 31
                    and (epi != 1 or (N % 2 == 0 and (N // 2) % 128 == 0)))
        if N % bn:
            return False
        if epi == 1 and (N % 2 or (N // 2) % (bn // 2)):
            return False
        return True

    def default_cfg(self, M: int) -> int:
        return 1 if M <= 64 else 0

    def _lookup(self, M: int, N: int, K: int, epi: int) -> Optional[Tuple[int, int]]:
        """Table choice at M, else at the nearest measured M above (same projection shape)."""
        ms = self.rows.get((N, K, epi))
        if not ms:
            return None
        at = bisect.bisect_left(ms, M)
        return self.table[(ms[at], N, K, epi)] if at < len(ms) else None

    def choose(self, M: int, N: int, K: int, epi: int) -> Optional[Tuple[int, int]]:
        """(tile configuration, split-K) of the hand kernel, or None for the library path."""
        if self.mode == "0":
            return None
        if self.mode == "force":
            for cfg in (self.default_cfg(M),) + tuple(range(N_CFGS)):
                for split in ((self.force_split, 1) if self.force_split > 1 else (1,)):
                    if self.supported(cfg, M, N, K, epi, split):
                        return (cfg, split)
            return None
        choice = self._lookup(M, N, K, epi)
        if choice is None and epi in (0, 2):
            # the store and residual epilogues run the same tile loop: a shape measured with one
            # (e.g. the TP row-parallel o / down projections, tuned with the residual epilogue
            # but called with the store epilogue before the fused all-reduce) takes that choice
            choice = self._lookup(M, N, K, 2 - epi)
        if choice is not None:
            return choice if choice[0] >= 0 and self.supported(choice[0], M, N, K, epi, choice[1]) else None
        if M > self.max_m or self.table:  # a measured table exists: unlisted shapes stay on the library
            return None
        cfg = self.default_cfg(M)
        return (cfg, 1) if self.supported(cfg, M, N, K, epi) else None

    def mid(self, M: int, N: int, K: int, epi: int) -> Optional[int]:
        """Plan of the kernel for tens to hundreds of rows (csrc/kernels/gemm_mid.hip), None where it is not taken: by its own rule, which rests on a
        model of its time, and where the table holds the projection and what stood there is faster from a row count up to the entry's
        (``tools/tune_hand_gemm.py --one-round``, up to seven row counts of each of 302 entries; 15 are listed, by 5 to 15 %: 256 x 2560 x 5120 21.0
        us against 25.2, but 193 rows 20.4 against 18.4, so from 214 on).  Decode steps of the 8b and 14b models bear out 7168 x 5120 at 49 to 64
        rows (0.5 to 2 us a layer) and 4096 x 12288 at 161 to 192 (3 to 6 us); not 7168 x 5120 at 33 to 40 and 97 to 128 (1.03 of the table's time
        alone, in steps 2.5 to 5 us a layer faster) and past 352, nor 4096 x 4096 and 5120 x 5120 into a residual past 640 (level)."""
        if self.mode != "1" or self.lib is None:
            return None
        if self.kept:
            ms = self.rows.get((N, K, epi), [])
            at = bisect.bisect_left(ms, M)
            if at < len(ms) and M >= self.kept.get((ms[at], N, K, epi), M + 1):
                return None
        p = self.lib.bcg_gemm_mid_plan(epi, M, N, K, 0)
        return p if p >= 0 else None

    def _rest(self, M: int, N: int, K: int, epi: int) -> Optional[Tuple[int, int]]:
        """The choice for the rows behind whole rounds."""
        p = self.mid(M, N, K, epi)
        return self.choose(M, N, K, epi) if p is None else (MID_CFG, p)

    def columns(self, M: int, N: int, K: int) -> int:
        """Gated projections (epilogue 1) below LARGE_M rows: how many of the N columns run as whole rounds of 256 x 256
        tiles, the others behind them; N: no split.

        A decode step's rows make few tiles, and one round and a sixteenth costs two: 448 x 34816 x 5120 (272 tiles) took 217
        us, as one round (125) and the last 2048 columns in 224 tiles of 64 x 64 (35) 165 to 172; 352 rows 175 -> 162, 512: 195 -> 176;
        768 x 22528 x 5120: 186 -> 162.  Taken where the rounds are at least 0.94 full, the rest is at most one small
        tile per CU (0.43 us per 64 of K against 1.46 for a round) and the rows fill 0.65 of their tiles (300 x 33792 x
        4096: 126 -> 129).  The one-round kernel takes the rest where it can (2048 columns of 5120 over 448 rows: 37 -> 27.6 us in the step)."""
        if self.mode != "1" or not 256 < M < LARGE_M or N % 256 or not self.supported(W4_CFG, M, N, K, 1):
            return N
        n_t, m_t = N // 256, -(-M // 256)
        rounds, rest = divmod(m_t * n_t, CUS)
        n1 = rounds * CUS // m_t
        if not (rounds and rest) or n1 * m_t < 0.94 * rounds * CUS or M < 0.65 * 256 * m_t:
            return N
        N2 = N - 256 * n1
        if -(-M // 64) * (N2 // 64) > CUS or not self.supported(SMALL_CFG, M, N2, K, 1):
            return N
        return 256 * n1

    def clamped_tiles(self, M: int, N: int, K: int) -> bool:
        """Whether the 256 x 256 kernel takes a clamped gated projection, the unit in its epilogue, from 512 rows on.

        The rule of the other gated epilogue, `_large_tiles`.  Product and activation pass over the one launch: filled rounds
        (0.8 and more) 16384 x 2048 (N x K) 1.13 to 1.29 over 1000 to 12000 rows, 24576 x 4096 1.00 to 1.13, 8192 x 1024 1.30 to 1.40; below
        that 0.75 (0.56 filled, 24576 x 4096, 640 rows) to 1.16."""
        return (self.mode == "1" and M >= 512 and self.supported(W4_CFG, M, N, K, 1)
                and self._large_tiles(K, 1, -(-M // 256) * (N // 256)))

    def tail_tiles(self, M: int, N: int, K: int, at: int) -> bool:
        """Whether the 256 x 256 kernel takes a projection whose columns from `at` on go through gelu in its epilogue.

        Product (as `pieces` has it) and activation pass over the one launch, from 1024 rows on: rounds filled to 0.9 and more 1.03 to
        1.18 (18432 x 4096 in 504 tiles: 1.00), to 0.8 up to K = 2048 1.01 to 1.14 (N 6656 and 11264), at K = 4096 0.92 to 1.01; below
        that 0.79 to 1.19."""
        if not (self.mode == "1" and M >= 1024 and 0 < at < N and at % 256 == 0 and self.supported(W4_CFG, M, N, K, 0)):
            return False
        tiles = -(-M // 256) * -(-N // 256)
        return tiles >= (0.8 if K <= 2048 else 0.9) * CUS * -(-tiles // CUS)

    def pieces(self, M: int, N: int, K: int, epi: int) -> List[Tuple[int, Optional[Tuple[int, int]]]]:
        """[(rows, choice)]: how the M rows run, one choice for all of them or two runs of rows.

        A prefill step has any number of rows, the table a few, and 256 x 256 tiles come in rounds of 256 (one per CU):
        288 tiles cost two rounds.  At row counts that the table does not hold, from LARGE_M on:
        * a last round that is short goes to the rows it is made of: (nearly) whole rounds for the first M1 rows, and the
          rest as a GEMM of its own, where that is estimated below 0.6 of a round (4449 x 4096 x 12288, us: library
          658, one 256 x 256 launch 470, split here 345).  `_main` says which kernel takes the rounds;
        * otherwise the 256 x 256 kernel takes all rows where `_large_tiles` says so (8183 x 11264 x 2048: library 369 us, here 301;
          2619 x 16384 x 2048: 167 and 149)."""
        choice = self.choose(M, N, K, epi)
        if self.mode != "1" or M < LARGE_M or (M, N, K, epi) in self.table or not self.supported(W4_CFG, M, N, K, epi):
            return [(M, choice)]
        n_t, m_t = -(-N // 256), -(-M // 256)
        tiles = m_t * n_t
        rounds, rest = divmod(tiles, CUS)
        if rounds and rest:
            m1 = rounds * CUS // n_t
            M1, M2 = 256 * m1, M - 256 * m1
            if (0 < m1 < m_t and m1 * n_t >= 0.94 * rounds * CUS
                    and 12 + 2e-6 * M2 * N * K / 0.8e3 < 0.6 * W4_KTILE_US * K / 64):
                split, main = self._main(N, K, epi, rounds, m1 * n_t, tiles)
                if (M1, N, K, epi) in self.table:
                    split, main = True, self.choose(M1, N, K, epi)
                if split:
                    return [(M1, main), (M2, self._rest(M2, N, K, epi))]
        if choice is None and self._large_tiles(K, epi, tiles):
            choice = (W4_CFG, 1)
        return [(M, choice)]

    @staticmethod
    def _even(tiles: int) -> bool:
        """Whether `tiles` tiles of 256 x 256 are the same number for every round that they take.

        The library's measured rate has two levels, and this tells them apart up to LONG_K: 6144 x 4096 (N x K), 7678 rows (720
        tiles, 3 rounds of 240) 1505 TFLOP/s, 4096 x 4096, 11612 rows (736 tiles) 904; the 256 x 256 kernel 1330 and 1415."""
        return tiles % -(-tiles // CUS) == 0

    @staticmethod
    def _main(N: int, K: int, epi: int, rounds: int, tiles: int, all_tiles: int) -> Tuple[bool, Optional[Tuple[int, int]]]:
        """(whether to split, the kernel of the rounds) for `tiles` of `all_tiles` tiles that fill `rounds` rounds but for a few.

        Library on all rows over the split, geometric mean (points slower by over 3 %), over 150 weights (N 256 to 20480, K 768 to
        18000) at 2048 to 12288 rows that the rules were not drawn from, 1591 splits: 1.22 (61), the slowest 0.81:
        * rounds of the same number of tiles go to the library: 1 round 1.33 (9 of 283), 2: 1.32 (0 of 226), 3: 1.24 (0 of 115), more 1.12
          (8 of 154), the 256 x 256 kernel 3 to 9 % less; but for one round of N not a multiple of 256 (1.42 against 1.30), and from LONG_K on
          up to 3 rounds (4 and more that are not exactly full: 0.90 to 1.1);
        * others go to the 256 x 256 kernel, the library being slow there (0.72 to 0.95): 3 rounds 1.13 (7 of 129), more 1.05 to
          1.09 (23 of 304); not 2 where all rows are even (1.00, 12 of 26), nor past 7 rounds (LONG_K: 5), 0.92 to 1.00;
        * the gated epilogue saves the library a pass: 1.07 to 1.26 (2 of 127)."""
        if epi == 1:
            return True, (W4_CFG, 1)
        if GemmPlan._even(tiles):
            if N % 256 and rounds == 1:
                return True, (W4_CFG, 1)
            return K < LONG_K or rounds <= 3 or tiles % CUS == 0, None
        if rounds == 2 and N % 256 == 0 and GemmPlan._even(all_tiles):
            return False, None
        return rounds <= (7 if K < LONG_K else 5), (W4_CFG, 1)

    @staticmethod
    def _large_tiles(K: int, epi: int, tiles: int) -> bool:
        """Whether the 256 x 256 kernel takes the library's place on all rows.

        Library over 256 x 256 kernel (points slower by over 3 %) over the same held-out points:
        * tiles that are uneven over their rounds: 2 rounds 1.45 (10 of 204), 3: 1.28 (6 of 538), 4: 1.15 (7 of 337), 5: 1.10 (43 of
          416), 6 to 8 1.07 (21 of 402); less filled ones and more rounds 0.87 to 1.06;
        * even ones: the library, 0.75 to 0.96; from LONG_K on its rate follows the rounds less, 2 rounds 1.30 (42 of 206), 3: 1.22 (4
          of 129), 4: 1.09 (11 of 94) between these fillings;
        * the gated epilogue: rounds filled to 0.8 and more 1.08 to 1.48 (0 of 402), to 0.65 up to K = 2048 1.06 to 1.15 (1 of 49), to
          0.55 up to K = 1024 1.19 to 1.53 (0 of 12), both from a full round on; below that 0.86 to 1.04."""
        rounds = -(-tiles // CUS)
        filled = tiles / (CUS * rounds)
        if epi == 1:
            return filled >= (0.8 if rounds == 1 or K > 2048 else 0.65 if K > 1024 else 0.55)
        if not GemmPlan._even(tiles):
            return filled >= (0.76 if rounds <= 3 else 0.8 if rounds <= 5 else 0.9) and rounds <= (8 if K < LONG_K else 6)
        return K >= LONG_K and 2 <= rounds <= 4 and 0.8 <= filled < (0.9 if K < 12000 else 0.95)


FP8_TABLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "engine", "tuned",
                         "hand_gemm_fp8.json")
FP8_RULE_MAX_M = 128  # unmeasured shapes: the hand fp8 kernel up to this M (it won every measured M <= 128)


class Fp8Plan:
    """Which fp8 projection GEMM runs: the hand block-scaled MFMA kernel (gemm.hip, F8) or
    hipBLASLt's ``torch._scaled_mm``.  Measured shapes (``engine/tuned/hand_gemm_fp8.json``,
    ``tools/bench_fp8_gemm.py``): the choice at the nearest measured M >= M, the library
    beyond the largest measured M; unmeasured shapes: the hand kernel up to FP8_RULE_MAX_M."""

    def __init__(self, tiles: Dict[int, Tuple[int, int]], table: Optional[str] = FP8_TABLE):
        self.tiles = tiles
        self.table: Dict[Tuple[int, int, int], Tuple[int, int]] = {}
        if table and os.path.exists(table):
            with open(table) as fh:
                for key, ch in json.load(fh).get("choice", {}).items():
                    self.table[tuple(map(int, key.split(",")))] = tuple(ch)

    def choose(self, M: int, N: int, K: int) -> Optional[Tuple[int, int]]:
        if os.environ.get("BCG_HAND_GEMM", "1") == "0" or K % 128 or M <= 0:
            return None
        above = [m for (m, n, k) in self.table if (n, k) == (N, K) and m >= M]
        if above:
            cfg, split = self.table[(min(above), N, K)]
        elif any((n, k) == (N, K) for (_, n, k) in self.table) or M > FP8_RULE_MAX_M:
            return None
        else:
            cfg, split = (6 if M <= 32 else 1 if M <= 64 else 0), 1
        if cfg < 0 or cfg not in self.tiles or K // 128 < split:
            return None
        if cfg == PP_CFG:  # 256 x 256 ping-pong fp8 kernel (prefill M): N % 16, 32-bit buffer offsets
            ok = N % 16 == 0 and M * K < 1 << 32 and N * K < 1 << 32 and 2 * (M + 256) * N < 1 << 31
        elif cfg == W4_CFG:  # four-wave 256 x 256 fp8 kernel: N % 16, offsets below 2 GiB
            ok = (N % 16 == 0 and (M + 256) * K < 1 << 31 and (N + 256) * K < 1 << 31
                  and 2 * (M + 256) * N < 1 << 31)
        else:
            ok = N % self.tiles[cfg][1] == 0
        return (cfg, split) if ok else None
