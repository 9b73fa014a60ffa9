"""The kernel for tens to hundreds of rows (csrc/kernels/gemm_mid.hip): every tile and split at sizes where it can go wrong, against a product in
float32; the plan over the sizes that it takes (CPU)."""

import ctypes
import os
import random

import pytest
import torch

from byzantine_consensus_llm_agents_amd.ops.gemm_plan import MID_CFG, GemmPlan
from byzantine_consensus_llm_agents_amd.utils.build import kernels_target

# (row blocks, column blocks) of the tiles, in the kernel's order
TILES = [(3, 1), (3, 2), (3, 3), (3, 4), (3, 6), (4, 2), (4, 3), (4, 4), (4, 5), (5, 4), (5, 5), (5, 6), (6, 4), (6, 6), (8, 4), (8, 5),
         (4, 8), (4, 10), (6, 8), (6, 10), (8, 6), (8, 10), (10, 6), (10, 8), (10, 12), (12, 10), (14, 8), (16, 8)]
TOL = 4e-3   # one rounding to bf16 of the result: 2^-9 relative, 0.58 of it on average; sums of 32 bits add less than 1e-5


@pytest.fixture(scope="module")
def ops():
    from byzantine_consensus_llm_agents_amd.ops import get_ops
    return get_ops("hip")


@pytest.fixture(scope="module")
def ops_cpu():
    if not os.path.exists(kernels_target()):
        pytest.skip("kernels not built")
    from byzantine_consensus_llm_agents_amd.ops.hip import hip_ops
    return hip_ops()


def _err(a, b):
    return ((a.float() - b).norm() / b.norm()).item()


def _run(ops, plan, epi, x, w, out, bias=None, residual=None, scales=(None, None)):
    lib, tiles = ops.library, ctypes.c_int()
    (M, K), N = x.shape, w.shape[0]
    ws = torch.empty(max(1, lib.bcg_gemm_mid_parts(plan, epi, M, N, ctypes.byref(tiles))), device="cuda")
    cnt = torch.zeros(max(1, tiles.value), dtype=torch.int32, device="cuda")
    ptr = [None if t is None else ctypes.c_void_p(t.data_ptr()) for t in (x, w, *scales, bias, residual, out, ws, cnt)]
    assert lib.bcg_gemm_mid(plan, epi, *ptr, M, N, K, N // 2, torch.cuda.current_stream().cuda_stream) == 0
    assert not cnt.any()
    return out


# rows: one, a tile's last, its first of a second one; columns not a multiple of the tile; K in 128-byte blocks of a row: one, odd and even numbers of
# them, parts of unequal length and of one block, as many parts as a plan may have (the last workgroup adds four at a time)
def _sizes(tile):
    mt, nt = TILES[tile]
    return ((1, 16, 1, 1), (16 * mt, 16 * nt, 5, 1), (16 * mt + 1, 32 * nt + 16, 11, 3), (16 * mt - 7, 16 * nt + 32, 17, 2),
            (16 * mt, 32 * nt, 10, 6), (16 * mt + 3, 16 * nt + 16, 16, 8), (5, 32, 8, 8))


@pytest.mark.gpu
@pytest.mark.parametrize("f8", [False, True], ids=["bf16", "fp8"])
@pytest.mark.parametrize("tile", range(len(TILES)), ids=[f"{16 * m}x{16 * n}" for m, n in TILES])
def test_every_tile(ops, tile, f8):
    torch.manual_seed(tile)
    for M, N, blocks, split in _sizes(tile):
        K = blocks * (128 if f8 else 64)
        x = torch.randn(M, K, device="cuda").bfloat16()
        w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
        bias, res = torch.randn(N, device="cuda").bfloat16(), torch.randn(M, N, device="cuda").bfloat16()
        scales, plan = (None, None), tile | split << 8
        y = x.float() @ w.float().t()
        if f8:
            x, w = x.to(torch.float8_e4m3fn), (w * 8).to(torch.float8_e4m3fn)
            scales = torch.rand(M, device="cuda") + 0.5, (torch.rand(N, device="cuda") + 0.5) / 8
            y = x.float() @ w.float().t() * scales[0][:, None] * scales[1]
        nan = lambda n: torch.full((M, n), float("nan"), dtype=torch.bfloat16, device="cuda")   # noqa: E731
        assert _err(_run(ops, plan, 0, x, w, nan(N), scales=scales), y) < TOL
        assert _err(_run(ops, plan, 0, x, w, nan(N), bias=bias, scales=scales), y + bias.float()) < TOL
        assert _err(_run(ops, plan, 2, x, w, res.clone(), residual=res, scales=scales), y + res.float()) < TOL
        if N % 32 == 0 and TILES[tile][1] % 2 == 0 and not f8:
            want = torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
            assert _err(_run(ops, plan, 1, x, w, nan(N // 2)), want) < TOL


# NaN in the bytes behind every operand's end, infinities and NaN in rows of x: nobody else's result changes
@pytest.mark.gpu
@pytest.mark.parametrize("f8", [False, True], ids=["bf16", "fp8"])
@pytest.mark.parametrize("tile,split", [(0, 1), (2, 3), (7, 1), (13, 8), (16, 2), (24, 1)])
def test_non_finite(ops, tile, split, f8):
    (mt, nt), K = TILES[tile], 128 * 9
    torch.manual_seed(tile)
    M, N = 16 * mt + 5, 32 * nt + 16
    dtype = torch.float8_e4m3fn if f8 else torch.bfloat16

    def behind(t):     # a copy that lies in front of NaN
        whole = torch.full((t.shape[0] + 300, *t.shape[1:]), float("nan"), device="cuda").to(t.dtype)
        whole[:len(t)] = t
        return whole[:len(t)]
    x, w = torch.randn(M, K, device="cuda").to(dtype), torch.randn(N, K, device="cuda").to(dtype)
    bias, res = torch.randn(N, device="cuda").bfloat16(), torch.randn(M, N, device="cuda").bfloat16()
    scales = (torch.rand(M, device="cuda"), torch.rand(N, device="cuda")) if f8 else (None, None)
    bad = [0, 16 * mt - 1, M - 1]
    xb = x.clone()
    xb.view(torch.uint8 if f8 else torch.int16)[bad[0], 3] = 0x7f if f8 else 0x7fc0
    xb.view(torch.uint8 if f8 else torch.int16)[bad[1], K - 1] = 0x7f if f8 else 0x7f80
    xb.view(torch.uint8 if f8 else torch.int16)[bad[2]] = 0x7f if f8 else 0x7fc0
    good = torch.ones(M, dtype=torch.bool, device="cuda")
    good[bad] = False
    for epi in (0, 1, 2):
        if epi == 1 and (f8 or nt % 2):
            continue
        n = (N - 16) if epi == 1 else N
        wn = w[:n].contiguous()
        kw = {0: {"bias": bias}, 1: {}, 2: {"residual": res}}[epi]
        want = _run(ops, tile | split << 8, epi, x, wn, torch.empty(M, n // 2 if epi == 1 else n, dtype=torch.bfloat16, device="cuda"), scales=scales, **kw)
        out = torch.full((M + 300, want.shape[1]), 7., dtype=torch.bfloat16, device="cuda")
        _run(ops, tile | split << 8, epi, behind(xb), behind(wn), out[:M], scales=tuple(s if s is None else behind(s) for s in scales),
             **{k: behind(v) for k, v in kw.items()})
        assert torch.equal(out[:M][good], want[good]) and want.isfinite().all()
        assert not out[:M][~good].isfinite().all(-1).any() and (out[M:] == 7).all()


# (tile, row tiles, column tiles, parts): row tiles of a column tile on two XCDs in some columns; the last one partly filled; K in parts
@pytest.mark.gpu
@pytest.mark.parametrize("tile,m_tiles,n_tiles,split", [(22, 3, 75, 1), (22, 3, 25, 3), (0, 5, 50, 1), (7, 2, 9, 1), (14, 3, 7, 6), (1, 7, 1, 1)])
def test_equal_rows_have_equal_results(ops, tile, m_tiles, n_tiles, split):
    (mt, nt), K = TILES[tile], 4096
    torch.manual_seed(tile)
    M, N = 16 * mt * m_tiles - 13, 16 * nt * n_tiles
    x = torch.randn(1, K // 2, device="cuda").bfloat16().repeat(M, 2)
    w = torch.randn(N, K // 2, device="cuda").bfloat16().repeat(1, 2)
    w[:, K // 2:].neg_()       # the sums are 0 but for what the order of their terms rounds
    out = _run(ops, tile | split << 8, 0, x, w, torch.empty(M, N, dtype=torch.bfloat16, device="cuda"))
    assert (out == out[:1]).all() and 0 < out.abs().max() < 1e-2


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(33, 2048, 1152), (100, 2048, 1152), (1024, 2048, 1152), (1025, 2048, 1152), (1536, 2048, 1152),
                                   (90, 544, 192), (400, 32, 4096)])
def test_entry_points_take_it_and_replay(ops, M, N, K):
    """A captured sequence of the three entry points, replayed on other inputs with eager calls between, gives what eager calls give; the operands
    that the library has to see do not come here."""
    torch.manual_seed(M)
    x, res = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(M, N, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    ops.prepare_device("cuda")
    assert ops.gemm_plan.mid(M, N, K, 0) is not None

    def step(r):
        return ops.linear(x, w), ops.linear_silu(x, w), ops.linear_residual(x, w, r)
    step(res.clone())
    r = res.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step(r)
    for _ in range(3):
        x.normal_()
        r.copy_(res)
        want = [t.clone() for t in step(res.clone())]
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        assert _err(want[0], x.float() @ w.float().t()) < TOL
    xg = x.clone().requires_grad_()
    ops.linear(xg, w).sum().backward()
    assert xg.grad is not None


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(33, 1040, 1024), (100, 4096, 1152), (176, 6144, 6144), (1000, 1024, 4096), (40, 2048, 8192)])
def test_fp8_entry_points_take_it(ops, M, N, K):
    torch.manual_seed(M)
    xq, wq = (torch.randn(n, K, device="cuda").to(torch.float8_e4m3fn) for n in (M, N))
    xs, ws = torch.rand(M, 1, device="cuda") + 0.5, (torch.rand(N, device="cuda") + 0.5) * K ** -0.5
    bias, res = torch.randn(N, device="cuda").bfloat16(), torch.randn(M, N, device="cuda").bfloat16()
    y = xq.float() @ wq.float().t() * xs * ws
    log = ops.dispatch_log
    log.enabled, log.calls, was = True, {}, (log.enabled, log.calls)
    try:
        got = ops.linear_fp8(xq, xs, wq, ws, bias), ops.linear_fp8(xq, xs, wq, ws), ops.linear_fp8_residual(xq, xs, wq, ws, res.clone())
        assert {(key[3], key[5].split("x")[0]) for key in log.calls} == {(0, str(MID_CFG)), (2, str(MID_CFG))}
    finally:
        log.enabled, log.calls = was
    for a, b in zip(got, (y + bias.float(), y, y + res.float())):
        assert _err(a, b) < TOL


@pytest.mark.gpu
def test_streams_and_captures_without_preparation(ops):
    """Split products on two streams at once don't share arrival counters, and a capture needs nothing prepared."""
    from byzantine_consensus_llm_agents_amd.ops import hip
    torch.manual_seed(0)
    M, N, K = 40, 1024, 8192
    x, w = torch.randn(M, K, device="cuda").bfloat16(), (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    own = getattr(hip.hip_ops, "__wrapped__", hip.hip_ops)()     # an instance that holds no counters yet
    assert own.gemm_plan.mid(M, N, K, 0) >> 8 > 1
    want = x.float() @ w.float().t()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = own.linear(x, w)
    for _ in range(2):
        graph.replay()
    assert _err(got, want) < TOL
    streams, outs = [torch.cuda.Stream() for _ in range(2)], []
    for _ in range(20):
        for s in streams:
            with torch.cuda.stream(s):
                outs.append(own.linear(x, w))
        outs.append(own.linear(x, w))
    torch.cuda.synchronize()
    assert all(torch.equal(o, outs[0]) for o in outs) and _err(outs[0], want) < TOL


@pytest.mark.gpu
@pytest.mark.parametrize("pool", [False, True], ids=["own pools", "one pool"])
def test_graphs_have_counters_of_their_own(ops, monkeypatch, pool):
    """Graphs captured on one stream (`torch.cuda.graph` takes the same for all) are replayed on several at once: no two may count arrivals in the same
    place, and none where eager products do.  Graphs that share a pool are replayed in turn.  One product of a graph is on a side stream."""
    torch.manual_seed(0)
    M, N, K = 40, 1024, 8192
    xs = [torch.randn(M, K, device="cuda").bfloat16() for _ in range(3)]
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    assert ops.gemm_plan.mid(M, N, K, 0) >> 8 > 1
    counters, launch = [], ops.library.bcg_gemm_mid
    monkeypatch.setattr(ops.library, "bcg_gemm_mid", lambda *a: counters.append(a[10].value) or launch(*a))
    want = [ops.linear(x, w) for x in xs]
    eager, graphs, outs, side = set(counters), [], [], torch.cuda.Stream()
    assert len(eager) == 1
    for x in xs:
        graphs.append(torch.cuda.CUDAGraph())
        counters.clear()
        with torch.cuda.graph(graphs[-1], pool=graphs[0].pool() if pool and len(graphs) > 1 else None):
            y = [ops.linear(x, w) for _ in range(2)]
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                y.append(ops.linear(x, w))
            torch.cuda.current_stream().wait_stream(side)
        outs.append(y)
        assert counters[0] == counters[1] != counters[2]
        assert pool or not eager & set(counters)
        eager |= set(counters)
    monkeypatch.undo()
    streams = [torch.cuda.Stream() for _ in graphs]
    for _ in range(10):
        for y in outs:
            for t in y:
                t.fill_(float("nan"))
        torch.cuda.synchronize()
        for g, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                g.replay()
                if not pool:
                    g.replay()
            if pool:
                s.synchronize()
        eagerly = ops.linear(xs[0], w)
        torch.cuda.synchronize()
        assert torch.equal(eagerly, want[0])
        assert all(torch.equal(t, u) for y, u in zip(outs, want) for t in y)


def test_plan_takes_one_round_and_refuses_the_rest():
    if not os.path.exists(kernels_target()):
        pytest.skip("kernels not built")
    lib = ctypes.CDLL(kernels_target())
    lib.bcg_gemm_mid_parts.restype = ctypes.c_int64
    rng, taken = random.Random(0), 0
    for _ in range(3000):
        M, N, K, epi, f8 = rng.randint(1, 2500), 8 * rng.randint(1, 5000), 32 * rng.randint(1, 600), rng.randrange(3), rng.randrange(2)
        p = lib.bcg_gemm_mid_plan(epi, M, N, K, f8)
        if p < 0:
            continue
        taken += 1
        assert 33 <= M <= (1024 if f8 else 1536) and (M <= 1024 or N > 512) and N % (32 if epi == 1 else 16) == 0 and K % (128 if f8 else 64) == 0 and not (f8 and epi == 1)
        mt, nt = TILES[p & 255]
        assert epi != 1 or nt % 2 == 0
        tiles = ctypes.c_int()
        floats = lib.bcg_gemm_mid_parts(p, epi, M, N, ctypes.byref(tiles))
        assert tiles.value == -(-M // (16 * mt)) * -(-N // (16 * nt)) and tiles.value * (p >> 8) <= 256
        assert floats == (0 if p >> 8 == 1 else tiles.value * (p >> 8) * 256 * mt * nt)
        assert K * (1 if f8 else 2) // 128 >= (p >> 8)
    assert taken > 50
    assert GemmPlan().mid(100, 4096, 4096, 0) is None     # (no library: no plan)
    plan = GemmPlan(lib)
    assert plan._rest(300, 4096, 4096, 0)[0] == MID_CFG
    for bad in ((0, 32, 4096, 4096, 0), (0, 1537, 4096, 4096, 0), (0, 1025, 4096, 4096, 1), (0, 1025, 512, 4096, 0), (0, 100, 4096, 4100, 0), (0, 100, 4104, 4096, 0), (1, 100, 4112, 4096, 0),
                (0, 100, 4096, 64, 0), (0, 100, 4096, 128, 0), (0, 100, 512, 192, 0), (0, 100, 512, 1024, 1), (0, 1024, 151936, 5120, 0), (1, 100, 4096, 4096, 1)):
        assert lib.bcg_gemm_mid_plan(*bad) == -1, bad
    # where the others are faster: both sides of each line
    for left, taken in (((0, 100, 16384, 64, 0), (1, 100, 16384, 64, 0)), ((0, 128, 16384, 128, 0), (0, 129, 16384, 128, 0)),
                        ((0, 300, 16384, 64, 0), (2, 300, 16384, 64, 0)), ((2, 128, 144, 2240, 0), (2, 129, 144, 2240, 0)),
                        ((0, 128, 144, 2240, 0), (0, 128, 144, 2304, 0)), ((0, 100, 128, 2240, 0), (0, 100, 160, 2240, 0)),
                        ((0, 100, 128, 2240, 0), (1, 100, 128, 2240, 0)), ((0, 300, 8192, 128, 1), (2, 300, 8192, 128, 1)),
                        ((0, 65, 8192, 256, 1), (0, 64, 8192, 256, 1)), ((0, 256, 4096, 256, 1), (0, 257, 4096, 256, 1)),
                        ((0, 200, 15360, 2048, 1), (0, 176, 15360, 2048, 1)), ((0, 200, 15360, 2048, 1), (2, 200, 15360, 2048, 1)),
                        ((0, 300, 4096, 3584, 1), (0, 300, 4096, 3712, 1)), ((0, 178, 4096, 2176, 1), (0, 178, 3968, 2048, 1))):
        assert lib.bcg_gemm_mid_plan(*left) == -1 and lib.bcg_gemm_mid_plan(*taken) >= 0, (left, taken)
    # what the table holds as faster is left too, from the row count that it says on up to its own
    assert plan.kept and all(key in plan.table and lib.bcg_gemm_mid_plan(key[3], rows, *key[1:3], 0) >= 0 and rows <= key[0] and
                             not any(rows <= m < key[0] for m in plan.rows[key[1:]]) for key, rows in plan.kept.items())
    for M, want in ((64, True), (65, True), (213, True), (214, False), (256, False), (257, True), (266, True), (267, False), (320, False),
                    (321, True), (458, True), (459, False), (512, False), (513, True)):
        assert (plan.mid(M, 2560, 5120, 0) is not None) == want, M
    assert plan.mid(256, 2560, 5120, 2) is not None and GemmPlan(lib, table=None).mid(256, 2560, 5120, 0) is not None


def test_few_rows_that_stay():
    """33 to 64 rows: the few-row kernel keeps small W and whole turns past 4096 columns, else the one-round kernel has them."""
    from byzantine_consensus_llm_agents_amd.ops.hip import few_rows_stay
    for M, N, K, gated, want in ((40, 1024, 2560, False, True), (40, 6144, 3072, False, True), (48, 6144, 3072, False, True), (49, 6144, 3072, False, False),
                                 (40, 6144, 4096, False, True), (40, 6144, 4608, True, False), (40, 4096, 3072, False, False), (40, 4096, 3072, True, True),
                                 (40, 8192, 2048, True, False), (40, 6144, 2176, True, False), (40, 6144, 1536, True, False)):
        assert few_rows_stay(M, N, K, gated) == want, (M, N, K, gated)


def test_gemm_nt_refuses_the_configuration(ops_cpu):
    """`gemm_nt` takes the tiles that `GemmPlan.supported` knows: the one-round kernel's number is none of them, whatever `out` and `bias` are."""
    x, w = torch.zeros(100, 4096).bfloat16(), torch.zeros(4096, 4096).bfloat16()
    plan = ops_cpu.gemm_plan.mid(100, 4096, 4096, 0)
    assert plan is not None and not ops_cpu.gemm_plan.supported(MID_CFG, 100, 4096, 4096, 0, plan)
    for kw in ({}, {"out": torch.zeros(1, 4096).bfloat16()}, {"bias": torch.zeros(1).bfloat16(), "out": torch.zeros(100, 4096).bfloat16()}):
        with pytest.raises(ValueError):
            ops_cpu.gemm_nt(x, w, (MID_CFG, plan), **kw)
