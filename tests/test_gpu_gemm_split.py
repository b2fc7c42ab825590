"""GPU: the GEMM tiles whose fp32 products are summed from bf16 parts, on the
inputs where the parts can fall short of fp32.

Every op, both tile sizes, rows with and without 16-byte alignment; the
kernel each shape takes is checked, so that a change of the cost model cannot
move a shape to another one unseen.
"""
import numpy as np
import pytest

import pitorch_amd as pa
from tests.test_gpu_gemm import bound_ok, ints, split_tile_call

pytestmark = pytest.mark.gpu

# op, M, N, K, accumulate, padding columns, tile
TILES = [(2, 1024, 2048, 768, 1, 0, 64), (2, 333, 2001, 701, 0, 1, 64), (0, 1024, 768, 2048, 1, 4, 64),
         (0, 501, 517, 1003, 1, 0, 64), (1, 2048, 768, 1000, 1, 0, 64), (1, 1003, 517, 501, 0, 3, 64),
         (2, 200, 32000, 300, 1, 4, 128), (2, 381, 21001, 301, 1, 2, 128), (0, 700, 12000, 260, 0, 4, 128),
         (0, 699, 12001, 261, 1, 0, 128), (1, 32000, 388, 300, 1, 0, 128), (1, 16003, 769, 301, 1, 2, 128)]
U = 2.0 ** -24


def on_tile(op, M, N, K, acc, pad, tile):
    return pa.gemm_plan(op, M, N, K, pad=pad, accumulate=acc)[:3] == (tile, tile, 0)


@pytest.mark.parametrize("op,M,N,K,acc,pad,tile", TILES)
def test_integer_products_are_exact(op, M, N, K, acc, pad, tile):
    assert on_tile(op, M, N, K, acc, pad, tile)
    A, B = ints((M, K), 61), ints((K, N), 62)
    C0 = ints((M, N), 63) if acc else np.full((M, N), np.nan, np.float32)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(split_tile_call(op, A, B, C0, M, N, K, acc, pad), (ref + C0 if acc else ref).astype(np.float32))


def one_term(op, M, N, K, pad, left, right, seed):
    """Products of one term each, `left` x `right` numbers, from either side: exact in
    64 bits, so what fp32 gives is their rounding."""
    rng = np.random.default_rng(seed)
    C0 = np.zeros((M, N), np.float32)
    A, B = left(rng, (M, K)), np.zeros((K, N), np.float32)
    at, sc = rng.integers(0, K, N), right(rng, N)
    B[at, np.arange(N)] = sc
    yield split_tile_call(op, A, B, C0, M, N, K, 0, pad), A[:, at].astype(np.float64) * sc
    A, B = np.zeros((M, K), np.float32), left(rng, (K, N))
    at, sc = rng.integers(0, K, M), right(rng, M)
    A[np.arange(M), at] = sc
    yield split_tile_call(op, A, B, C0, M, N, K, 0, pad), B[at].astype(np.float64) * sc[:, None]


def spread(lo, hi):
    """Numbers of all 24 bits (fewer below 2^-126), of exponents lo .. hi-1 and either sign."""
    return lambda rng, shape: (rng.uniform(1, 2, shape) * rng.choice((-1, 1), shape) * 2.0 ** rng.integers(lo, hi, shape)).astype(np.float32)


def powers(lo, hi):
    return lambda rng, shape: (2.0 ** rng.integers(lo, hi, shape)).astype(np.float32)


# bf16 reaches down to 2^-133: the third part of a number below 2^-109 can
# lie below it.  Down to the smallest subnormal; the products are normal.
@pytest.mark.parametrize("op,M,N,K,acc,pad,tile", TILES)
@pytest.mark.parametrize("lo,hi", [(-149, -100), (-126, -108), (-112, -60)])
def test_small_operands_keep_their_bits(op, M, N, K, acc, pad, tile, lo, hi):
    assert on_tile(op, M, N, K, 0, pad, tile)
    for got, exact in one_term(op, M, N, K, pad, spread(lo, hi), powers(60, 100), K + lo):
        assert np.array_equal(got, exact.astype(np.float32))


# Subnormal products: fp32's spacing there is 2^-149.
@pytest.mark.parametrize("op,M,N,K,acc,pad,tile", TILES)
def test_subnormal_products(op, M, N, K, acc, pad, tile):
    assert on_tile(op, M, N, K, 0, pad, tile)
    for got, exact in one_term(op, M, N, K, pad, spread(-74, -64), spread(-72, -64), K):
        assert np.all(np.abs(got - exact) <= 2.0 ** -150 * 1.001)


# The operands whose parts' dropped products are largest, just above 1 + 2^-8.  One
# term: the three dropped are below U(1 + 2^-8) of the product, the last of the six sums is off by
# at most one spacing (2U), the ones before it are of at most 2^-7 of it.
@pytest.mark.parametrize("op,M,N,K,acc,pad,tile", TILES)
def test_one_term_of_the_worst_bits(op, M, N, K, acc, pad, tile):
    assert on_tile(op, M, N, K, 0, pad, tile)
    worst = lambda rng, shape: (1 + 2.0 ** -8 + rng.integers(-2 ** 9, 2 ** 9, shape) * 2.0 ** -23 + rng.choice((0, 2.0 ** -7), shape)).astype(np.float32)
    for got, exact in one_term(op, M, N, K, pad, worst, worst, K):
        assert np.max(np.abs(got - exact) / exact) <= U * (3 + 2.0 ** -4)


# The same in short sums: as many roundings as terms, as in fp32 (K < 16 runs there).
@pytest.mark.parametrize("op,M,N,tile", [(2, 1024, 8192, 128), (2, 300, 20001, 128), (1, 17248, 669, 128), (0, 1024, 8192, 128)])
@pytest.mark.parametrize("K", [1, 2, 3, 7, 15, 16, 17])
def test_short_sums_round_as_fp32(op, M, N, tile, K):
    assert on_tile(op, M, N, K, 1, 0, tile)
    rng = np.random.default_rng(K)
    A, B = ((1 + 2.0 ** -8 + rng.integers(-2 ** 9, 2 ** 9, s) * 2.0 ** -23).astype(np.float32) for s in ((M, K), (K, N)))
    got = split_tile_call(op, A, B, np.zeros((M, N), np.float32), M, N, K, 1, 0)
    a, b = A.astype(np.float64), B.astype(np.float64)
    assert bound_ok(got, a @ b, np.abs(a) @ np.abs(b), K)


@pytest.mark.parametrize("op,M,N,K,acc,pad,tile", TILES)
def test_non_finite(op, M, N, K, acc, pad, tile):
    """Infinities, NaNs and numbers next to the largest, as a product and sum in
    fp32 gives them; the other rows and columns as ever."""
    assert on_tile(op, M, N, K, 0, pad, tile)
    rng = np.random.default_rng(M)
    A, B = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(0.5, 1, (K, N)).astype(np.float32)
    A[3, 5], A[17, K - 1], A[M - 1, 0] = np.inf, -np.inf, np.nan
    A[9, 2], A[10, 2], A[10, 3] = np.finfo(np.float32).max, np.inf, -np.inf
    B[2, 7] = 0.25
    got = split_tile_call(op, A, B, np.zeros((M, N), np.float32), M, N, K, 0, pad)
    assert np.all(np.isposinf(got[3])) and np.all(np.isneginf(got[17]))
    assert np.all(np.isnan(got[M - 1])) and np.all(np.isnan(got[10]))
    clean = np.setdiff1d(np.arange(M), (3, 10, 17, M - 1))
    a, b = A[clean].astype(np.float64), B.astype(np.float64)
    assert bound_ok(got[clean], a @ b, np.abs(a) @ np.abs(b), K)
