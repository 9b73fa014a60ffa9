"""Which projections of a few rows the streaming kernel takes (`few_rows_pay`): both sides of its lines.  No GPU."""
from byzantine_consensus_llm_agents_amd.ops.hip import SKINNY_ROW_BYTES, SKINNY_ROWS, few_rows_pay


def test_lines():
    pay = lambda M, N, K, gated=False: few_rows_pay(M, N, 2 * K, gated)
    assert all(pay(M, N, K) for M in (1, 16) for N in (256, 5120, 151936) for K in (896, 5120, 12288))
    assert not pay(4, 256, 16384) and pay(4, 512, 16384) and not pay(16, 1024, 14336) and pay(16, 1536, 17408) and pay(16, 256, 17408)
    assert not pay(10, 3072, 16384, True) and pay(10, 4096, 16384, True)
    assert pay(20, 5120, 5120) and not pay(20, 2048, 6144) and pay(32, 4096, 17408) and not pay(24, 512, 768) and pay(24, 512, 768, True)
    assert pay(31, 1024, 4096) and not pay(32, 1024, 4096) and pay(32, 1536, 4096) and not pay(32, 2048, 2560) and not pay(17, 256, 1536)
    assert pay(48, 8192, 2048) and not pay(48, 8736, 2048) and not pay(40, 2048, 8192) and not pay(40, 1536, 3072) and pay(40, 2048, 3072)
    assert not pay(40, 2048, 2560) and pay(40, 3072, 2560) and not pay(40, 8192, 4096) and not pay(36, 1024, 448) and pay(36, 768, 768)
    assert pay(64, 4096, 2048) and not pay(64, 4096, 4096) and pay(64, 2048, 2048, True) and not pay(64, 768, 1024)
    assert pay(64, 1024, 896) and not pay(64, 1024, 448) and not pay(49, 3072, 1536) and pay(49, 4096, 1536)


def test_every_size_has_an_answer():
    for M in range(1, SKINNY_ROWS + 1):
        for N in (8, 260, 1000, 4096, 8192, 8200, 200000):
            for row_bytes in range(128, SKINNY_ROW_BYTES + 1, 1920):
                for gated in (False, True):
                    assert few_rows_pay(M, N, row_bytes, gated) in (True, False)
