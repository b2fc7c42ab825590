"""GPU parity of the fp32 MFMA training GEMMs against the oracle.

* integer-valued inputs (1..16): every product and partial sum is exact in
  fp32 (|sum| < 2^24), so GPU == oracle BIT FOR BIT for any summation order —
  this also pins the MFMA operand/result lane layout;
* U(-1,1) inputs: |C - C_fp64| <= gamma_K * (|A||B|) elementwise (the fp32
  forward-error bound for a K-term dot product).
Shapes: the reference's GEMM unit-test sizes (dev/tests/gemm/test_gemm.c:
82-83) and every training GEMM of the 15M config at T=256 (R=255).
"""
import numpy as np
import pytest

import pitorch_amd as pa
from pitorch_amd._hip import DeviceArray
from tests._oracle import P, oracle
from tests.test_oracle import lcg_ints

pytestmark = pytest.mark.gpu
R = 255
DW = [(288, 288), (768, 288), (288, 768), (32000, 288)]      # dW[out,in] += dY^T X, K = R
DX = [(288, 288), (768, 288), (288, 768), (32000, 288)]      # dX[R,in] = dY[R,out] W[out,in], K = out


def ints(shape, seed):
    return np.random.default_rng(seed).integers(1, 17, shape).astype(np.float32)


def bound_ok(C, A64_B64_exact, absAB, K):
    gamma = K * 2.0 ** -24 / (1 - K * 2.0 ** -24)
    return np.all(np.abs(C - A64_B64_exact) <= gamma * absAB + 1e-30)


@pytest.mark.parametrize("n", [16, 32])
def test_sgemm_square_exact(n):
    A = lcg_ints(n * n, 42, 16).reshape(n, n)
    B = lcg_ints(n * n, 137, 16).reshape(n, n)
    C = np.zeros((n, n), np.float32)
    L = pa.load_ptmi()
    assert L.ptmi_sgemm_rect(P(A), P(B), P(C), n, n, n, 0) == 0
    ref = np.zeros((n, n), np.float32)
    oracle().po_sgemm(P(A), P(B), P(ref), n, n, n)
    assert np.array_equal(C, ref)


@pytest.mark.parametrize("out_dim,in_dim", DW)
def test_backward_weight_batched_exact(out_dim, in_dim):
    dY, X = ints((R, out_dim), 1), ints((R, in_dim), 2)
    dW = ints((out_dim, in_dim), 3)
    ref = dW.copy()
    L = pa.load_ptmi()
    assert L.ptmi_matmul_backward_weight_batched_checked(P(dW), P(dY), P(X), out_dim, in_dim, R) == 0
    oracle().po_matmul_backward_weight_batched(P(ref), P(dY), P(X), out_dim, in_dim, R)
    assert np.array_equal(dW, ref)
    # the void entry with the reference's exact signature (pt_train.c:475-477)
    L.ptmi_matmul_backward_weight_batched(P(dW), P(dY), P(X), out_dim, in_dim, R)
    oracle().po_matmul_backward_weight_batched(P(ref), P(dY), P(X), out_dim, in_dim, R)
    assert np.array_equal(dW, ref)


# T = 1: the rank-1 matmul_backward_weight (pitorch/train/pt_backward_ops.c:
# 43-49), unit-tested by the reference at 32x16 (dev/tests/train/
# test_backward_ops.c:86-105); also the config-5 projection shapes.
@pytest.mark.parametrize("out_dim,in_dim", [(32, 16), (288, 288), (768, 288), (288, 768), (32000, 288), (5, 3)])
def test_backward_weight_rank1_exact(out_dim, in_dim):
    dy, x = ints(out_dim, 11), ints(in_dim, 12)
    dW = ints((out_dim, in_dim), 13)
    ref = dW.copy()
    L = pa.load_ptmi()
    L.ptmi_matmul_backward_weight_batched(P(dW), P(dy), P(x), out_dim, in_dim, 1)
    oracle().po_matmul_backward_weight(P(ref), P(dy), P(x), out_dim, in_dim)
    assert np.array_equal(dW, ref)


# sgemm_rect_tmu's own call site (matmul_backward_weight_gpu,
# pitorch/train/pt_train.c:536-543): C[V,D] += A[V,R] . X[R,D] with
# M = 32000, K = R = 255, N = D = 288, accumulate = 1, num_qpus = 12; and
# the rect shapes below, all integer-exact against the oracle's
# sgemm_rect_tmu restatement.
@pytest.mark.parametrize("M,K,N,acc", [(32000, 255, 288, 1), (255, 288, 288, 0), (255, 32000, 288, 1),
                                       (300, 77, 130, 1), (1, 5, 3, 0), (100, 3001, 70, 1), (1000, 301, 900, 0)])
def test_sgemm_rect_tmu_exact(M, K, N, acc):
    A, B = ints((M, K), M + 1), ints((K, N), K + 2)
    C = ints((M, N), N + 3) if acc else np.zeros((M, N), np.float32)
    ref = C.copy()
    L = pa.load_ptmi()
    L.ptmi_sgemm_rect_tmu(P(A), P(B), P(C), M, K, N, 12, acc)
    oracle().po_sgemm_rect(P(A), P(B), P(ref), M, K, N, acc)
    assert np.array_equal(C, ref)


@pytest.mark.parametrize("n", [16, 32])
def test_sgemm_cpu_signature_exact(n):
    """ptmi_sgemm_cpu: sgemm_cpu's signature (pitorch/ops/gemm/gemm.h:19-20),
    at the reference's test sizes (dev/tests/gemm/test_gemm.c:82-83)."""
    A = lcg_ints(n * n, 7, 16).reshape(n, n)
    B = lcg_ints(n * n, 9, 16).reshape(n, n)
    C = np.full((n, n), np.nan, np.float32)
    L = pa.load_ptmi()
    L.ptmi_sgemm_cpu(P(A), P(B), P(C), n, n, n)
    ref = np.zeros((n, n), np.float32)
    oracle().po_sgemm(P(A), P(B), P(ref), n, n, n)
    assert np.array_equal(C, ref)


@pytest.mark.parametrize("out_dim,in_dim", DX)
def test_backward_input_batched_exact(out_dim, in_dim):
    dY, W = ints((R, out_dim), 4), ints((out_dim, in_dim), 5)
    dX = np.zeros((R, in_dim), np.float32)
    L = pa.load_ptmi()
    assert L.ptmi_matmul_backward_input_batched(P(dX), P(W), P(dY), out_dim, in_dim, R, 0) == 0
    ref = np.zeros((R, in_dim), np.float32)
    for t in range(R):
        oracle().po_matmul_backward_input(P(ref[t]), P(W), P(dY[t]), out_dim, in_dim)
    assert np.array_equal(dX, ref)


# Kernel paths: 32x32 tiles (255x288x288, 300x77x130, 1x5x3), 64x64 bf16-product
# tiles (1000x301x900), the same with split K (K = 3001 and 32000).
@pytest.mark.parametrize("M,K,N", [(255, 288, 288), (255, 32000, 288), (300, 77, 130), (1, 5, 3), (100, 3001, 70),
                                   (1000, 301, 900)])
def test_sgemm_rect_random_bounded(M, K, N):
    rng = np.random.default_rng(M + K + N)
    A = rng.uniform(-1, 1, (M, K)).astype(np.float32)
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    C0 = rng.uniform(-1, 1, (M, N)).astype(np.float32)
    C = C0.copy()
    L = pa.load_ptmi()
    assert L.ptmi_sgemm_rect(P(A), P(B), P(C), M, K, N, 1) == 0
    exact = C0.astype(np.float64) + A.astype(np.float64) @ B.astype(np.float64)
    assert bound_ok(C, exact, np.abs(C0) + np.abs(A) @ np.abs(B), K + 1)


@pytest.mark.parametrize("op", [0, 1, 2])
def test_gemm_dev_ops_with_strides(op):
    """Device-pointer entry: NN, TN, NT with padded leading dimensions."""
    rng = np.random.default_rng(op)
    M, N, K = 200, 96, 130
    pad = 4
    if op == 0:
        A = rng.uniform(-1, 1, (M, K + pad)); B = rng.uniform(-1, 1, (K, N + pad))
        Aop, Bop = A[:, :K], B[:, :N]
    elif op == 1:
        A = rng.uniform(-1, 1, (K, M + pad)); B = rng.uniform(-1, 1, (K, N + pad))
        Aop, Bop = A[:, :M].T, B[:, :N]
    else:
        A = rng.uniform(-1, 1, (M, K + pad)); B = rng.uniform(-1, 1, (N, K + pad))
        Aop, Bop = A[:, :K], B[:, :K].T
    A, B = A.astype(np.float32), B.astype(np.float32)
    C = np.zeros((M, N + pad), np.float32)
    dA, dB, dC = DeviceArray.from_host(A), DeviceArray.from_host(B), DeviceArray.from_host(C)
    L = pa.load_ptmi()
    assert L.ptmi_gemm_dev(op, dA.ptr, A.shape[1], dB.ptr, B.shape[1], dC.ptr, N + pad, M, N, K, 0, None) == 0
    assert L.ptmi_sync() == 0
    got = dC.download().reshape(M, N + pad)
    exact = Aop.astype(np.float32).astype(np.float64) @ Bop.astype(np.float32).astype(np.float64)
    absab = np.abs(Aop.astype(np.float32)) @ np.abs(Bop.astype(np.float32))
    assert bound_ok(got[:, :N], exact, absab, K)
    assert np.all(got[:, N:] == 0)          # padding columns untouched
    for a in (dA, dB, dC):
        a.free()


# Grids of 768 blocks and more take their tiles in XCD order (each XCD a
# contiguous tile range, ordered along the larger operand), the bf16-product
# tiles' always do: ragged M, N and K on 64x64 and 128x128 tiles, split K for the
# NN forms; a NaN-filled C shows any tile left unwritten.
@pytest.mark.parametrize("op,M,N,K", [(2, 200, 20000, 300), (2, 260, 20000, 300), (0, 255, 320, 30000),
                                      (0, 130, 288, 30000), (1, 30004, 288, 130), (1, 32000, 256, 131)])
def test_gemm_dev_large_grids(op, M, N, K):
    rng = np.random.default_rng(M + N + K)
    if op == 0:
        A = rng.uniform(-1, 1, (M, K)); B = rng.uniform(-1, 1, (K, N))
        Aop, Bop = A, B
    elif op == 1:
        A = rng.uniform(-1, 1, (K, M)); B = rng.uniform(-1, 1, (K, N))
        Aop, Bop = A.T, B
    else:
        A = rng.uniform(-1, 1, (M, K)); B = rng.uniform(-1, 1, (N, K))
        Aop, Bop = A, B.T
    A, B = A.astype(np.float32), B.astype(np.float32)
    dA, dB = DeviceArray.from_host(A), DeviceArray.from_host(B)
    dC = DeviceArray.from_host(np.full((M, N), np.nan, np.float32))
    L = pa.load_ptmi()
    assert L.ptmi_gemm_dev(op, dA.ptr, A.shape[1], dB.ptr, B.shape[1], dC.ptr, N, M, N, K, 0, None) == 0
    assert L.ptmi_sync() == 0
    got = dC.download().reshape(M, N)
    Af, Bf = Aop.astype(np.float32).astype(np.float64), Bop.astype(np.float32).astype(np.float64)
    assert bound_ok(got, Af @ Bf, np.abs(Af) @ np.abs(Bf), K)
    for a in (dA, dB, dC):
        a.free()


# The largest outputs (4M elements and more), NT and TN: on 128x128 bf16-product
# tiles, and on the direct-to-LDS fp32 tiles (TN, K = 7): integer-exact at the
# classifier shapes of config 5, with and without accumulate, and on ragged M, N and K.
@pytest.mark.parametrize("op,M,N,K,acc", [(2, 256, 32000, 288, 0), (2, 256, 32000, 288, 1), (2, 193, 21845, 36, 1),
                                          (1, 32000, 288, 255, 0), (1, 32000, 288, 255, 1), (1, 16388, 260, 7, 0)])
def test_gemm_dev_direct_lds_exact(op, M, N, K, acc):
    if op == 1:
        A, B = ints((K, M), 21), ints((K, N), 22)
        ref = A.T.astype(np.float64) @ B.astype(np.float64)
    else:
        A, B = ints((M, K), 23), ints((N, K), 24)
        ref = A.astype(np.float64) @ B.T.astype(np.float64)
    C0 = ints((M, N), 25) if acc else np.full((M, N), np.nan, np.float32)
    if acc:
        ref = ref + C0
    dA, dB, dC = DeviceArray.from_host(A), DeviceArray.from_host(B), DeviceArray.from_host(C0)
    L = pa.load_ptmi()
    assert L.ptmi_gemm_dev(op, dA.ptr, A.shape[1], dB.ptr, B.shape[1], dC.ptr, N, M, N, K, acc, None) == 0
    assert L.ptmi_sync() == 0
    got = dC.download().reshape(M, N)
    assert np.array_equal(got, ref.astype(np.float32))
    for a in (dA, dB, dC):
        a.free()


# The per-layer NT GEMMs with at most 9 K steps per split take the panel
# kernel (every K tile of the split in flight): integer-exact at the
# config-5 forward shapes (K split 4 ways at K = 768, summed by the split-K
# reduction), with accumulate, and on ragged M, N and K.
@pytest.mark.parametrize("M,N,K,acc", [(256, 864, 288, 0), (256, 288, 288, 1), (256, 1536, 288, 0),
                                       (256, 288, 768, 1), (255, 100, 100, 0), (33, 31, 4, 1), (70, 2050, 284, 0)])
def test_gemm_dev_panel_nt_exact(M, N, K, acc):
    A, B = ints((M, K), 31), ints((N, K), 32)
    ref = A.astype(np.float64) @ B.T.astype(np.float64)
    C0 = ints((M, N), 33) if acc else np.full((M, N), np.nan, np.float32)
    if acc:
        ref = ref + C0
    dA, dB, dC = DeviceArray.from_host(A), DeviceArray.from_host(B), DeviceArray.from_host(C0)
    L = pa.load_ptmi()
    assert L.ptmi_gemm_dev(2, dA.ptr, K, dB.ptr, K, dC.ptr, N, M, N, K, acc, None) == 0
    assert L.ptmi_sync() == 0
    got = dC.download().reshape(M, N)
    assert np.array_equal(got, ref.astype(np.float32))
    for a in (dA, dB, dC):
        a.free()


# Middle and large GEMMs, mostly on the bf16-product tiles (64x64 with K dealt to
# four waves, 128x128 for many tiles; tests/test_gpu_gemm_split.py holds each of
# them): whole and ragged M, N and K, K ranges that leave a wave without work,
# split K, rows without 16-byte alignment, padded leading dimensions, accumulate.
SPLIT_TILES = [(0, 1024, 768, 2048, 0, 0), (1, 770, 2050, 1000, 1, 2), (2, 1024, 2048, 768, 1, 0), (2, 333, 8001, 701, 0, 0),
               (0, 501, 517, 1003, 1, 0), (1, 1003, 517, 501, 0, 1), (0, 65, 4100, 4097, 0, 3), (2, 200, 32000, 300, 1, 0),
               (1, 33000, 130, 300, 0, 0), (2, 257, 21847, 37, 0, 0), (0, 700, 12000, 260, 0, 4), (2, 64, 65600, 20, 0, 0)]


def split_tile_call(op, A, B, C0, M, N, K, acc, pad):
    """C (+)= op(A).op(B) of dense A [M,K], B [K,N] through ptmi_gemm_dev,
    operands stored as `op` wants them with `pad` NaN columns after each row."""
    def stored(x):
        return np.ascontiguousarray(np.pad(x, ((0, 0), (0, pad)), constant_values=np.nan), np.float32)
    a, b, c = stored(A.T if op == 1 else A), stored(B.T if op == 2 else B), stored(C0)
    dA, dB, dC = DeviceArray.from_host(a), DeviceArray.from_host(b), DeviceArray.from_host(c)
    L = pa.load_ptmi()
    assert L.ptmi_gemm_dev(op, dA.ptr, a.shape[1], dB.ptr, b.shape[1], dC.ptr, N + pad, M, N, K, acc, None) == 0
    assert L.ptmi_sync() == 0
    got = dC.download().reshape(M, N + pad)[:, :N]
    for d in (dA, dB, dC):
        d.free()
    return got


@pytest.mark.parametrize("op,M,N,K,acc,pad", SPLIT_TILES)
def test_gemm_dev_split_tiles_exact(op, M, N, K, acc, pad):
    A, B = ints((M, K), 41), ints((K, N), 42)
    C0 = ints((M, N), 43) if acc else np.full((M, N), np.nan, np.float32)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    got = split_tile_call(op, A, B, C0, M, N, K, acc, pad)
    assert np.array_equal(got, (ref + C0 if acc else ref).astype(np.float32))


@pytest.mark.parametrize("op,M,N,K,acc,pad", SPLIT_TILES)
def test_gemm_dev_split_tiles_keep_all_bits(op, M, N, K, acc, pad):
    """One operand random in all 24 bits over 60 binades, the other with one
    power of two per sum: every result is a single product and exact."""
    rng = np.random.default_rng(K)
    full = lambda shape: (rng.uniform(1, 2, shape) * 2.0 ** rng.integers(-30, 30, shape) * rng.choice((-1, 1), shape)).astype(np.float32)
    C0 = np.zeros((M, N), np.float32)
    A, B = full((M, K)), np.zeros((K, N), np.float32)
    at, sc = rng.integers(0, K, N), (2.0 ** rng.integers(-20, 20, N)).astype(np.float32)
    B[at, np.arange(N)] = sc
    assert np.array_equal(split_tile_call(op, A, B, C0, M, N, K, 0, pad), A[:, at] * sc)
    A, B = np.zeros((M, K), np.float32), full((K, N))
    at, sc = rng.integers(0, K, M), (2.0 ** rng.integers(-20, 20, M)).astype(np.float32)
    A[np.arange(M), at] = sc
    assert np.array_equal(split_tile_call(op, A, B, C0, M, N, K, 0, pad), B[at] * sc[:, None])


@pytest.mark.parametrize("op,M,N,K,acc,pad", [SPLIT_TILES[i] for i in (0, 3, 4, 7, 8)])
def test_gemm_dev_split_tiles_non_finite(op, M, N, K, acc, pad):
    """Infinities, NaNs and numbers next to the largest give what a product
    and sum in fp32 gives, and leave the other rows and columns alone."""
    rng = np.random.default_rng(M)
    A, B = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(0.5, 1, (K, N)).astype(np.float32)
    A[3, 5], A[17, K - 1], A[M - 1, 0] = np.inf, -np.inf, np.nan
    A[9, 2], A[10, 2], A[10, 3] = np.finfo(np.float32).max, np.inf, -np.inf
    B[2, 7] = 0.25
    C0 = np.zeros((M, N), np.float32)
    got = split_tile_call(op, A, B, C0, M, N, K, 0, pad)
    assert np.all(np.isposinf(got[3])) and np.all(np.isneginf(got[17]))
    assert np.all(np.isnan(got[M - 1])) and np.all(np.isnan(got[10]))
    clean = np.setdiff1d(np.arange(M), (3, 10, 17, M - 1))
    a, b = A[clean].astype(np.float64), B.astype(np.float64)
    assert bound_ok(got[clean], a @ b, np.abs(a) @ np.abs(b), K)


# Large outputs of short K on each of the kernels that take them (as
# tests/test_gemm_plan.py pins the choice), ragged in every size; C's padding
# columns are NaN before and after.
@pytest.mark.parametrize("op,M,N,K,acc,pad,kernel", [
    (2, 64, 65600, 1, 0, 0, (64, 64, 1)), (2, 63, 66601, 7, 1, 3, (64, 64, 1)), (2, 33, 131100, 96, 0, 4, (64, 64, 1)),
    (2, 300, 20001, 7, 1, 1, (128, 128, 0)), (2, 1024, 8192, 16, 0, 4, (128, 128, 0)), (0, 1023, 8191, 17, 1, 2, (128, 128, 0)),
    (1, 17247, 669, 41, 1, 3, (128, 128, 0)), (1, 32000, 132, 33, 1, 4, (128, 128, 0)), (1, 32004, 132, 31, 0, 4, (128, 96, 1)),
])
def test_gemm_dev_short_k(op, M, N, K, acc, pad, kernel):
    assert pa.gemm_plan(op, M, N, K, pad=pad, accumulate=acc)[:3] == kernel
    A, B = ints((M, K), 51), ints((K, N), 52)
    C0 = ints((M, N), 53) if acc else np.full((M, N), np.nan, np.float32)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    c = np.pad(C0, ((0, 0), (0, pad)), constant_values=np.nan)
    stored = [np.ascontiguousarray(np.pad(x, ((0, 0), (0, pad)), constant_values=np.nan))
              for x in (A.T if op == 1 else A, B.T if op == 2 else B)]
    dA, dB, dC = (DeviceArray.from_host(x) for x in (*stored, c))
    L = pa.load_ptmi()
    assert L.ptmi_gemm_dev(op, dA.ptr, stored[0].shape[1], dB.ptr, stored[1].shape[1], dC.ptr, N + pad, M, N, K, acc, None) == 0
    assert L.ptmi_sync() == 0
    got = dC.download().reshape(M, N + pad)
    assert np.array_equal(got[:, :N], (ref + C0 if acc else ref).astype(np.float32)) and np.all(np.isnan(got[:, N:]))
    for d in (dA, dB, dC):
        d.free()


@pytest.mark.parametrize("op,M,N,K", [(0, 512, 768, 2048), (0, 300, 512, 1536), (1, 700, 500, 1200)])
def test_gemm_dev_on_two_streams(op, M, N, K):
    """GEMMs on two streams of the caller and on the library's, all in flight
    at once: each is whole on the caller's streams, cut on the library's."""
    import ctypes
    from pitorch_amd._hip import hip
    L, H = pa.load_ptmi(), hip()
    assert pa.gemm_plan(op, M, N, K)[3] > 1 and pa.gemm_plan(op, M, N, K, callers_stream=1)[3] == 1
    assert L.ptmi_init(0) == 0
    streams = [ctypes.c_void_p(), ctypes.c_void_p()]
    for s in streams:
        assert H.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0             # hipStreamNonBlocking
    jobs = []
    for i, s in enumerate((*streams, None)):
        A, B = ints((K, M) if op == 1 else (M, K), 70 + i), ints((N, K) if op == 2 else (K, N), 80 + i)
        ref = (A.T if op == 1 else A).astype(np.float64) @ (B.T if op == 2 else B).astype(np.float64)
        jobs.append((s, A, B, DeviceArray.from_host(A), DeviceArray.from_host(B), DeviceArray(M * N), ref))
    for _ in range(20):
        for s, A, B, dA, dB, dC, _ref in jobs:
            assert L.ptmi_gemm_dev(op, dA.ptr, A.shape[1], dB.ptr, B.shape[1], dC.ptr, N, M, N, K, 0, s) == 0
    assert H.hipDeviceSynchronize() == 0
    for s, A, B, dA, dB, dC, ref in jobs:
        assert np.array_equal(dC.download().reshape(M, N), ref.astype(np.float32))
        for d in (dA, dB, dC):
            d.free()
    for s in streams:
        assert H.hipStreamDestroy(s) == 0


# More rows than one grid's 65535 tiles of 32: split_plan counts 64-row tiles
# for NT outputs of 4 Mi elements, and takes 65535 of those.
@pytest.mark.parametrize("acc", [0, 1])
def test_gemm_dev_most_rows(acc):
    M, N, K = 2200003, 2, 5
    assert pa.gemm_plan(2, M, N, K, accumulate=acc)[:3] == (32, 32, 1)
    A, B, C0 = ints((M, K), 91), ints((K, N), 92), ints((M, N), 93)
    ref = (A @ B + (C0 if acc else 0)).astype(np.float32)
    assert np.array_equal(split_tile_call(2, A, B, C0, M, N, K, acc, 0), ref)
    a = DeviceArray(16)
    assert pa.load_ptmi().ptmi_gemm_dev(2, a.ptr, K, a.ptr, K, a.ptr, N, 65535 * 64 + 1, N, K, 0, None) == 1
    assert b"M too large" in pa.load_ptmi().ptmi_last_error()
    a.free()


def test_gemm_errors():
    L = pa.load_ptmi()
    A = np.ones((4, 4), np.float32)
    assert L.ptmi_sgemm_rect(P(A), P(A), P(A), 0, 4, 4, 0) == 1
    assert L.ptmi_gemm_dev(3, P(A), 4, P(A), 4, P(A), 4, 4, 4, 4, 0, None) == 1
