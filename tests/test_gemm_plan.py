"""Which kernel a GEMM takes (CPU only: pure host arithmetic behind
ptmi_gemm_plan, no device call).

The kernels: 32x32 fp32 tiles, bf16 products on 64x64 and 128x128 tiles, and
two fp32 tiles for large outputs of short K (128x96 and 64x64).  The shapes are
ones where the kernel named here was the fastest on the MI355X, or within 3% of
it, so a change of the cost model that moves one of them needs a new
measurement.
"""
import random

import pytest

import pitorch_amd as pa

F32, F64, DL, B64, B128 = (32, 32, 1), (64, 64, 1), (128, 96, 1), (64, 64, 0), (128, 128, 0)


@pytest.mark.parametrize("op,M,N,K,acc,kernel", [
    # one short K step or a few into large outputs: what is left after the tile's own start counts
    (2, 64, 65600, 1, 0, F64), (2, 64, 65600, 20, 0, F64), (2, 64, 65600, 96, 1, F64), (2, 64, 65600, 128, 0, B64),
    (2, 1024, 8192, 16, 0, B128), (2, 1024, 8192, 64, 0, B128), (2, 300, 20001, 7, 0, B128), (2, 1024, 4096, 64, 0, B128),
    (2, 2048, 2049, 96, 0, B128), (2, 131, 32000, 64, 0, B128), (2, 400, 16000, 64, 0, B128),
    (1, 32000, 288, 16, 0, DL), (1, 32000, 288, 16, 1, B128), (1, 32000, 288, 64, 0, B128),
    (1, 17248, 669, 64, 1, B128), (0, 1024, 8192, 16, 0, B128),
    # ordinary training GEMMs
    (2, 1024, 2048, 768, 0, B64), (0, 1024, 768, 2048, 0, B64), (1, 2048, 768, 1024, 1, B64), (2, 1024, 32000, 768, 0, B128),
    (1, 32000, 768, 1024, 1, B128), (0, 1024, 768, 32000, 0, B64), (2, 256, 32000, 288, 0, B128), (2, 1024, 4096, 768, 0, B64),
    # small ones, and long K from few rows
    (2, 64, 768, 288, 0, F32), (0, 64, 288, 768, 0, F32), (1, 768, 288, 64, 1, F32), (0, 36, 160, 6725, 0, F32),
    (0, 16, 96, 31586, 0, F32), (0, 2048, 1024, 64, 0, F32),
])
def test_kernel_of_measured_shapes(op, M, N, K, acc, kernel):
    assert pa.gemm_plan(op, M, N, K, accumulate=acc)[:3] == kernel


def test_plans_hold_over_the_range():
    rng = random.Random(3)
    seen = set()
    for _ in range(4000):
        M, N, K = (int(2 ** rng.uniform(0, e)) for e in (15, 18, 15))
        op, acc, epi = rng.randrange(3), rng.randrange(2), rng.choice((0, 0, 0, 1, 2, 3))
        if epi:
            op, acc, N = 0 if epi == 3 else 2, 0, N + N % 2
        tm, tn, fp32, splits = pa.gemm_plan(op, M, N, K, accumulate=acc, epilogue=epi)
        seen.add((tm, tn, fp32))
        assert 1 <= splits <= 64
        if epi:
            assert splits == 1 and (tm, tn, fp32) in ((F32, B64) if epi == 1 else (F32, B64, B128))
        if splits > 1:                     # a piece is at least one K step, partials fit the workspace
            assert (K + splits - 1) // splits >= 32
            assert splits * M * N <= (64 << 20 if fp32 else 4 << 20)
        # rows too long for the bf16 tiles' 32-bit offsets
        assert pa.gemm_plan(op, M, N, K, pad=1 << 22, accumulate=acc, epilogue=epi)[2] == 1
    assert seen == {F32, F64, DL, B64, B128}


def test_calls_on_other_streams_share_no_workspace_they_did_not_need():
    """K is cut on a caller's stream only where the fp32 tiles cut it: 32x32
    tiles, fewer than 128 and K > 288, or K >= 4096 (and NT outputs of 4 Mi elements):
    fewer than 512 tiles of 64x64."""
    rng, cut = random.Random(4), 0
    tiles = lambda M, N, T: -(-M // T) * -(-N // T)
    for _ in range(6000):
        M, N, K = (int(2 ** rng.uniform(0, e)) for e in (12, 13, 15))
        op, acc = rng.randrange(3), rng.randrange(2)
        splits = pa.gemm_plan(op, M, N, K, accumulate=acc, callers_stream=1)[3]
        big = op == 2 and M * N >= 4 << 20
        may = tiles(M, N, 64) < 512 if K >= 4096 else not big and tiles(M, N, 32) < 128 and K > 288
        assert splits == 1 or may, (op, M, N, K)
        cut += splits > 1
        if may:                                          # nothing else differs from the library's stream
            assert pa.gemm_plan(op, M, N, K, accumulate=acc, callers_stream=1) == pa.gemm_plan(op, M, N, K, accumulate=acc)
    assert cut > 500
    for op, M, N, K in ((0, 512, 768, 2048), (0, 300, 512, 1536)):
        assert pa.gemm_plan(op, M, N, K)[3] > 1 and pa.gemm_plan(op, M, N, K, callers_stream=1)[3] == 1
