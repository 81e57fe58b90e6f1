"""The fp32 products formed from three-piece bf16 splits (csrc/gemm.hip), at the edges of their paths:
the 64 x 64, 64 x 128 and 128 x 128 tiles, whole pairs of 16-deep chunks (the branch-free loop) and
remainders, split K, K of one or two chunks, operands with no bf16 split (infinities, NaN, values past the largest bf16) and
values whose pieces underflow. Reference: the f64 product of the same fp32 values.

Bounds: the pairs of pieces left out are below 2^-24 of a term (2^-25 each of the two larger ones) and a
16-deep step rounds its sum a few times: 2^-23 (K / 4 + 8) of the sum of |terms| an element. That alone would let a missing pair
of small pieces (2^-17 of a term) pass at large K, so the 2-norm of the error is held to 5e-7 of the
result's too (8 to 64 such roundings give 6e-8 to 3e-7, one missing pair 2e-6).
"""
import numpy as np
import pytest

import talos_hip as th
from common import block_params, f32, gacha_states, mla_params, ppo_params
from test_gpu_models import block_slices, mla_slices, ppo_slices, run_block, run_mla, run_ppo

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
                                   (10240, 128, 64), (10247, 128, 40), (10300, 65, 31), (16383, 128, 33),
                                   (16384, 128, 64), (16391, 128, 40), (16400, 65, 31),  # 64 x 128 (tA = 0)
                                   (2048, 2048, 32), (2049, 2047, 48), (2100, 2048, 33),  # 128 x 128
                                   (2048, 2048, 64), (2049, 2047, 16), (2049, 2047, 17), (2112, 2048, 31)])
# (of the last two lines K <= 32 with A plain: 64 x 128, the width of several tiles)
def test_split_products(tA, tB, M, N, K):
    A, B = operands(tA, tB, M, N, K)
    got = product(tA, tB, A, B).astype(np.float64)
    ref, mag = exact(tA, tB, A, B)
    assert np.all(np.abs(got - ref) <= 2.0**-23 * (K / 4 + 8) * mag)
    assert np.linalg.norm(got - ref) <= 5e-7 * np.linalg.norm(ref)


@pytest.mark.parametrize("M,N,K", [(64, 64, 32), (70, 64, 40), (10247, 128, 32), (16391, 128, 32), (2049, 2048, 32),
                                   (2049, 2048, 64)])
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


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(70, 64, 40), (60, 70, 1100), (16391, 128, 40), (2049, 2047, 48), (150, 130, 70000)])
def test_infinity_in_any_layout(tA, tB, M, N, K):
    """One infinity in the last line of either operand: that line of C infinite, every other element as finite ones
    are (tiles without one by the split products, the line's tiles, in one K split of the long ones, by fp32 products:
    their 2-norm bound 2^-24 sqrt(K))."""
    for side in (0, 1):
        X = list(operands(tA, tB, M, N, K))
        line = X[side].T if side != (tA, tB)[side] else X[side]  # [M or N][K]
        line[-1, K - 1] = np.inf
        got = product(tA, tB, *X).astype(np.float64)
        rest = (slice(0, -1), slice(None)) if side == 0 else (slice(None), slice(0, -1))
        other = (X[1 - side].T if 1 - side != (tA, tB)[1 - side] else X[1 - side])[:, K - 1]
        assert np.array_equal(got[-1] if side == 0 else got[:, -1], np.inf * f32(other))
        line[-1, K - 1] = 0.0
        ref, mag = exact(tA, tB, *X)
        err = (got - ref)[rest]
        assert np.all(np.abs(err) <= (2.0**-23 * (K / 4 + 8) * mag)[rest])
        assert np.linalg.norm(err) <= 2.0**-24 * K**0.5 * np.linalg.norm(ref[rest])


def test_zero_times_infinity():
    A, B = operands(0, 0, 70, 64, 40)
    A[3, 5], B[5, 7] = np.inf, 0.0
    got = product(0, 0, A, B)
    assert np.isnan(got[3, 7]) and not np.any(np.isnan(np.delete(got, 3, 0)))


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(64, 64, 32), (70, 66, 40), (60, 70, 1100), (16391, 128, 40), (2048, 2048, 32),
                                   (2048, 2048, 64)])
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
@pytest.mark.parametrize("M,N", [(64, 64), (70, 33), (16391, 128), (2049, 2047)])
def test_one_product(tA, tB, M, N):
    """K = 1: every element is the fp32 product of its two operands, rounded once."""
    A, B = operands(tA, tB, M, N, 1)
    a, b = A.reshape(M, 1), B.reshape(1, N)
    assert np.array_equal(product(tA, tB, A, B), a * b)


# The fp32 products of whole plans with every epilogue that their tiles have (input norm, norm backward,
# bias gradients, GELU, row dots, column maps), on each tile size. Each weight gets values too small to split in
# every 32nd column of a row and every 32nd row of a column, so that every tile of it holds some, the
# inputs and output gradients in every 32nd column of every 16th token. They are far below a rounding of any
# result: the plan with zeros in their place, whose products are the split ones, computes the same. The two's
# errors against f64 add: 1e-5 of a tensor's 2-norm is ten times the larger (5.7e-7, the latent block at
# 64 x 256); one misplaced row of 32768 would be 5e-3.
def mark_weights(p, slices, cols, value):
    p = p.copy()
    for name, c in cols.items():
        w = p[slices[name]].reshape(-1, c)
        w[5, ::32] = value
        w[::32, min(7, c - 1)] = value
    return p


def mark_tokens(x, value):
    x = x.copy()
    x[:, ::16, ::32] = value
    return x


def check_same(got, ref, slices):
    for g, r, parts in zip(got, ref, slices):
        g, r = np.atleast_1d(f32(g)).reshape(-1), np.atleast_1d(f32(r)).reshape(-1)
        for name, sl in (parts or {"": slice(None)}).items():
            assert np.linalg.norm(g[sl] - r[sl]) <= 1e-5 * np.linalg.norm(r[sl]), name
    assert not np.array_equal(got[0], ref[0])  # (other products: other roundings)


TINY = np.float32(2.0**-120)


@pytest.mark.parametrize("B,S", [(8, 64), (184, 64), (512, 64)])
def test_block_by_fp32_products(B, S):
    d, F = 128, 512
    rng = np.random.default_rng(B)
    cfg, slices = th.BlockCfg(B, S, d, 4, 32, F, 1, th.ACT_GELU, 1e-6, 10000.0), block_slices(d, F)
    cols = {"wqkv": 3 * d, "wo": d, "w1": F, "w2": d}
    p = f32(block_params(rng, d, F, gain_jitter=True)).astype(np.float32)
    x, g = rng.standard_normal((2, B, S, d), dtype=np.float32)
    got, ref = (run_block(cfg, mark_weights(p, slices, cols, v), mark_tokens(x, v), mark_tokens(g, v))
                for v in (TINY, np.float32(0)))
    check_same(got, ref, (None, slices, None))


@pytest.mark.parametrize("B,S", [(2, 64), (16, 256), (64, 256)])
def test_latent_block_by_fp32_products(B, S):
    ci = [B, S, 512, 8, 128, 32, 64, 64, 0, 0]
    rng = np.random.default_rng(B)
    cols = {"W_dkv": 128, "W_uk": 512, "W_uv": 512, "W_q": 512, "W_kr": 256, "W_qr": 256, "W_o": 512}
    p = f32(mla_params(rng, ci)).astype(np.float32)
    x, g = rng.standard_normal((2, B, S, 512), dtype=np.float32)
    got, ref = (run_mla(ci, th.PREC_FP32, mark_weights(p, mla_slices(ci), cols, v), mark_tokens(x, v), mark_tokens(g, v))
                for v in (TINY, np.float32(0)))
    check_same(got, ref, (None, mla_slices(ci), None))


@pytest.mark.parametrize("B,S", [(40, 16), (700, 21), (4096, 32)])
def test_policy_by_fp32_products(B, S):
    d, F = 128, 512
    cfg = th.PpoCfg(B, S, 8, d, 2, 4, 32, F, 3, 1, th.ACT_GELU, 1e-5, 10000.0, 0.2, 0.5, 0.01)
    rng = np.random.default_rng(B)
    slices = ppo_slices(cfg)
    cols = {"We": d, "Wout": d, "Wa": 3, "Wc": 1}
    for layer in ("L0.", "L1."):
        cols.update({layer + "wqkv": 3 * d, layer + "wo": d, layer + "w1": F, layer + "w2": d})
    p = f32(ppo_params(rng, cfg)).astype(np.float32)
    batch = (gacha_states(rng, B, S).astype(np.float32), rng.integers(0, 3, B).astype(np.int32),
             *rng.standard_normal((2, B), dtype=np.float32), np.full(B, -1.1, np.float32))
    got, ref = (run_ppo(cfg, mark_weights(p, slices, cols, v), *batch) for v in (TINY, np.float32(0)))
    check_same(got[1:], ref[1:], (slices, None, None))


@pytest.mark.parametrize("M,N", [(64, 64), (16391, 128), (2048, 2048)])
@pytest.mark.parametrize("K", [16, 40, 512])
def test_largest_left_out_pairs(M, N, K):
    """1 + 2^-8 - 2^-17 = 1, 2^-8, -2^-17 in pieces: the pairs left out come to 3.97 * 2^-26 of each term, all of one
    sign. 2^-24 for them and two roundings of 2^-24 for each 16-deep step and the final sum."""
    v = np.float32(1 + 2.0**-8 - 2.0**-17)
    got = product(0, 0, np.full((M, K), v), np.full((K, N), -v)).astype(np.float64)
    ref = -K * float(v) ** 2
    assert np.all(np.abs(got - ref) <= 2.0**-24 * (1 + 2 * (-(-K // 16) + 1)) * -ref)


@pytest.mark.parametrize("draw", ["uniform", "normal", "absolute"])
@pytest.mark.parametrize("M,N,K", [(64, 64, 512), (16384, 128, 512), (4096, 4096, 512), (4096, 4096, 2048),
                                   (4096, 4096, 8192)])  # (K in one piece)
def test_no_less_accurate_than_fp32_products(M, N, K, draw):
    """Sums that grow with every term as well as zero-mean ones: the 2-norm of the error against that of the fp32
    products, which one value too small to split in every 32 rows of A (and far below any rounding) brings about."""
    rng = np.random.default_rng(K)
    A, B = ((rng.random(s, dtype=np.float32) if draw == "uniform" else rng.standard_normal(s, dtype=np.float32))
            for s in ((M, K), (K, N)))
    if draw == "absolute":
        A, B = np.abs(A), np.abs(B)
    A[::32, K // 2] = 0.0
    rows = np.linspace(1, M - 1, 48).astype(int)
    ref = f32(A[rows]) @ f32(B)
    split = np.linalg.norm(product(0, 0, A, B)[rows] - ref)
    A[::32, K // 2] = 2.0**-120
    assert split <= np.linalg.norm(product(0, 0, A, B)[rows] - ref)
