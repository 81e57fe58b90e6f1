"""The fp32 products formed from three-piece bf16 splits (csrc/gemm.hip), at the edges of their paths:
the 64 x 64, 64 x 128 and 128 x 128 tiles, whole pairs of 16-deep chunks (the branch-free loop) and
remainders, split K, operands with no bf16 split (infinities, NaN, values past the largest bf16) and
values whose pieces underflow. Reference: the f64 product of the same fp32 values.

Bounds: the pairs of pieces left out are below 3 * 2^-26 of a term and a 16-deep step rounds its sum a
few times: 2^-23 (K / 4 + 8) of the sum of |terms| an element. That alone would let a missing pair
of small pieces (2^-17 of a term) pass at large K, so the 2-norm of the error is held to 5e-7 of the
result's too (8 to 64 such roundings give 6e-8 to 3e-7, one missing pair 2e-6).
"""
import numpy as np
import pytest

import talos_hip as th
from common import f32

pytestmark = pytest.mark.gpu
DA = th.DeviceArray


def product(tA, tB, A, B):
    M, K = A.shape[::-1] if tA else A.shape
    N = B.shape[0] if tB else B.shape[1]
    dA, dB, dC = DA.from_numpy(A), DA.from_numpy(B), DA.zeros((M, N))
    th.call("talos_gemm_f32", tA, tB, M, N, K, 1.0, dA.ptr, A.shape[1], dB.ptr, B.shape[1], 0.0, dC.ptr, N, None)
    return dC.numpy()


def operands(tA, tB, M, N, K):
    rng = np.random.default_rng(M + 7 * N + 31 * K + 2 * tA + tB)
    return (rng.normal(size=(K, M) if tA else (M, K)).astype(np.float32),
            rng.normal(size=(N, K) if tB else (K, N)).astype(np.float32))


def exact(tA, tB, A, B):
    a, b = f32(A).T if tA else f32(A), f32(B).T if tB else f32(B)
    return a @ b, np.abs(a) @ np.abs(b)


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(64, 64, 32), (65, 63, 16), (1, 64, 17), (130, 96, 48), (60, 70, 5003),  # 64 x 64
                                   (10240, 128, 64), (10247, 128, 40), (10300, 65, 31),  # 64 x 128
                                   (2048, 2048, 32), (2049, 2047, 48), (2100, 2048, 33)])  # 128 x 128
def test_split_products(tA, tB, M, N, K):
    A, B = operands(tA, tB, M, N, K)
    got = product(tA, tB, A, B).astype(np.float64)
    ref, mag = exact(tA, tB, A, B)
    assert np.all(np.abs(got - ref) <= 2.0**-23 * (K / 4 + 8) * mag)
    assert np.linalg.norm(got - ref) <= 5e-7 * np.linalg.norm(ref)


@pytest.mark.parametrize("M,N,K", [(64, 64, 32), (70, 64, 40), (10247, 128, 32), (2049, 2048, 32)])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38, -3.4e38])
def test_values_without_a_split(M, N, K, value):
    A, B = operands(0, 0, M, N, K)
    B *= np.float32(0.01)  # (3.4e38 times the row stays finite)
    A[M - 1, K - 1] = value
    got = product(0, 0, A, B).astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref, mag = exact(0, 0, A, B)
    ok = np.isfinite(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    assert np.all(np.abs(got - ref)[ok] <= (2.0**-23 * (K / 4 + 8) * mag)[ok])


def test_zero_times_infinity():
    A, B = operands(0, 0, 70, 64, 40)
    A[3, 5], B[5, 7] = np.inf, 0.0
    got = product(0, 0, A, B)
    assert np.isnan(got[3, 7]) and not np.any(np.isnan(np.delete(got, 3, 0)))


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(64, 64, 32), (70, 66, 40), (60, 70, 1100), (10247, 128, 40), (2048, 2048, 32)])
@pytest.mark.parametrize("power", [-118, -128])
def test_third_piece_underflows(tA, tB, M, N, K, power):
    """Values near 2^-118, whose third piece bf16 cannot hold (2^-134 of an absolute error is 4e-6 of them, as a
    2-norm), and subnormal ones, whose second it cannot, are multiplied as fp32 values: either operand of
    them, or one line of it beside zeros. The 2-norm of K independent roundings of partial sums no larger than the
    result's 2-norm: 2^-24 sqrt(K)."""
    for small in (0, 1):
        for one_line in (False, True):
            X = list(operands(tA, tB, M, N, K))
            X[small] *= np.float32(2.0**power)
            X[1 - small] *= np.float32(2.0**60)
            if one_line:  # the last row of op(A) or column of op(B)
                line = X[small].T if small != (tA, tB)[small] else X[small]
                line[:-1] = 0.0
            got = product(tA, tB, *X).astype(np.float64)
            ref, mag = exact(tA, tB, *X)
            assert np.all(np.abs(got - ref) <= 2.0**-23 * (K / 4 + 8) * mag)
            assert np.linalg.norm(got - ref) <= 2.0**-24 * K**0.5 * np.linalg.norm(ref)


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N", [(64, 64), (70, 33), (10247, 128), (2049, 2047)])
def test_one_product(tA, tB, M, N):
    """K = 1: every element is the fp32 product of its two operands, rounded once."""
    A, B = operands(tA, tB, M, N, 1)
    a, b = A.reshape(M, 1), B.reshape(1, N)
    assert np.array_equal(product(tA, tB, A, B), a * b)
