"""linear_int8's streamed codes against float64: one row, the edges of the
32-row strips and of the 64- and 128-row blocks, ragged columns, K of one
phase (128), short of one, just past one and not a multiple of 16 (the last
codes of a row are loaded from further back), rows at odd addresses, one,
several and more than 32 K ranges, the sizes that the plan leaves to the tiles,
and scales of zero, infinity and NaN.  Each size names the plan it is meant
for.

Bar: A is kept to 16 bits and a sign (2^-17 of each value at most) and the
codes exactly; fp32 sums add about 1e-6: 1e-5 normwise."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(808)


def _run(gpu, x, q, s):
    return gpu.linear_int8(gpu.from_numpy(x), gpu.from_numpy(q), gpu.from_numpy(s)).to_numpy().astype(np.float64)


def _data(M, N, K):
    x = RNG.standard_normal((M, K)).astype(np.float32)
    q = RNG.integers(-128, 128, (N, K)).astype(np.int8)
    s = (RNG.random(N) * 0.02 + 1e-4).astype(np.float32)
    return x, q, s


def _plan(M, N, K):
    from applegpu_runtime._native import lib
    buf = ctypes.create_string_buffer(96)
    assert lib.applegpu_ffi_gemm_plan(M, N, K, 1, 3, True, True, buf, 96) == 0
    return buf.value.decode()


TILES = 0
SIZES = [  # rows, columns, k, ranges of k (0: the tiles)
    # one row strip: both ends of its k and rows, columns past a block's 256
    (1, 1, 128, 1), (1, 33, 129, 1), (3, 255, 143, 1), (16, 257, 256, 1), (7, 1000, 4099, 17), (31, 40, 8191, 22),
    (32, 256, 256, 1), (17, 300, 383, 3), (32, 2048, 512, 4), (1, 33, 127, TILES), (16, 8192, 112, TILES),
    (17, 257, 240, TILES), (5, 100, 16, TILES),
    # two strips: rows of both, k of few phases (ragged) and of many
    (33, 257, 193, 1), (64, 100, 383, 3), (65, 100, 999, 8), (128, 300, 201, 1), (129, 1, 1000, 8), (256, 77, 257, 3),
    (33, 40, 4096, 16), (64, 3072, 3072, 12), (64, 2048, 8192, 22), (65, 3073, 2048, 8), (128, 20, 8192, 32),
    (100, 9, 16001, 42), (256, 2049, 2048, 6), (200, 6144, 768, 2),
    (33, 257, 191, TILES), (64, 512, 256, TILES), (65, 512, 512, TILES), (128, 1024, 4096, TILES), (256, 768, 272, TILES),
    (256, 4096, 1024, TILES), (257, 300, 500, TILES), (200, 5, 3, TILES)]


@pytest.mark.parametrize("M,N,K,ranges", SIZES)
def test_against_float64(gpu, M, N, K, ranges):
    plan = _plan(M, N, K)
    if ranges == TILES:
        assert plan.startswith("mf"), plan
    else:
        assert plan == f"i8 stream 256 cols splits={ranges}", plan
    x, q, s = _data(M, N, K)
    got = _run(gpu, x, q, s)
    want = (x.astype(np.float64) @ q.astype(np.float64).T) * s.astype(np.float64)
    assert got.shape == want.shape
    # a single output may cancel: the roundings, independent, are compared with
    # the root of the terms' squares, which the norm of many outputs averages to
    size = np.sqrt((x.astype(np.float64) ** 2) @ (q.astype(np.float64) ** 2).T) * s
    assert np.linalg.norm(got - want) <= 1e-5 * max(np.linalg.norm(want), np.linalg.norm(size))
    np.testing.assert_array_equal(got, _run(gpu, x, q, s))


def test_whole_numbers_are_exact(gpu):
    """Small whole numbers are exact in A's hi half: a wrong place of any code
    or value shows."""
    for M, N, K in [(40, 70, 200), (40, 70, 203), (100, 300, 1001), (5, 256, 2048), (20, 40, 128)]:
        x = RNG.integers(-3, 4, (M, K)).astype(np.float32)
        q = RNG.integers(-128, 128, (N, K)).astype(np.int8)
        s = np.exp2(RNG.integers(-8, 8, N)).astype(np.float32)
        want = (x.astype(np.int64) @ q.astype(np.int64).T) * s.astype(np.float64)
        np.testing.assert_array_equal(_run(gpu, x, q, s), want)


def test_special_scales_and_rows(gpu):
    x, q, s = _data(20, 64, 300)
    s[3], s[5], s[7], s[9] = 0.0, np.inf, np.nan, -0.5
    x[4, 299] = np.nan
    got = _run(gpu, x, q, s)
    want = (x.astype(np.float64) @ q.astype(np.float64).T) * np.where(np.isfinite(s), s, np.nan).astype(np.float64)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.linalg.norm(got[ok] - want[ok]) <= 1e-5 * np.linalg.norm(want[ok])


@pytest.mark.parametrize("M,N,K", [(1, 40, 128), (20, 64, 300), (64, 512, 4096), (130, 256, 201), (64, 64, 64)])
def test_sums_past_fp32_before_the_scale(gpu, M, N, K):
    """Results that fp32 holds come out although the sum of values times codes
    passes its range on the way, in one range of K, in one of its halves or in
    the sum of both; a scale of zero gives zero."""
    x, q, s = _data(M, N, K)
    s[:] = (RNG.random(N) + 0.5) * 2.0 ** -20
    s[1 % N] = 0.0
    x *= 2.0 ** 118                                # 2^118 * 2^7 * sqrt(K) and more
    x[0, :16] = 2.0 ** 126
    q[:, :16] = 127
    got = _run(gpu, x, q, s)
    want = (x.astype(np.float64) @ q.astype(np.float64).T) * s.astype(np.float64)
    assert np.isfinite(got).all()
    assert np.linalg.norm(got / 2.0 ** 110 - want / 2.0 ** 110) <= 1e-5 * np.linalg.norm(want / 2.0 ** 110)
    assert (got[:, 1 % N] == 0).all()
    s[:] = 2.0 ** 20                               # and those that it does not hold are infinite
    q[:, :] = 127
    x[:] = 2.0 ** 118
    assert np.isposinf(_run(gpu, x, q, s)).all()
