"""linear_int8's streamed codes against float64: one row, the edges of the
32-row strips and of the 64- and 128-row blocks, ragged columns, K of one
phase (128), short of one, just past one and not a multiple of 16 (the last
codes of a row are loaded from further back), rows at odd addresses, one and
several K ranges, the sizes that the plan leaves to the tiles, and scales of
zero, infinity and NaN.

Bar: A is kept to 16 bits and a sign (2^-17 of each value at most) and the
codes exactly; fp32 sums add about 1e-6: 1e-5 normwise."""
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


@pytest.mark.parametrize("M,N,K", [(1, 1, 16), (1, 33, 17), (3, 255, 31), (32, 256, 128), (33, 257, 129), (64, 512, 256),
                                   (65, 100, 383), (128, 300, 127), (129, 1, 1000), (256, 768, 272), (7, 1000, 4099),
                                   (65, 2049, 2048),                                   (31, 40, 8191), (64, 2048, 8192), (200, 5, 3),  # K < 16: the tiles
                                   (65, 512, 512), (257, 300, 500)])  # few codes or many rows: the tiles
def test_against_float64(gpu, M, N, K):
    x, q, s = _data(M, N, K)
    got = _run(gpu, x, q, s)
    want = (x.astype(np.float64) @ q.astype(np.float64).T) * s.astype(np.float64)
    assert got.shape == want.shape
    # K = 16 .. 31 of one row or column: the per-value bound, not its average
    assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
    np.testing.assert_array_equal(got, _run(gpu, x, q, s))


def test_whole_numbers_are_exact(gpu):
    """Small whole numbers are exact in A's hi half: a wrong place of any code
    or value shows."""
    for M, N, K in [(40, 70, 200), (100, 300, 1001), (5, 256, 2048)]:
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


@pytest.mark.parametrize("M,N,K", [(1, 40, 128), (20, 64, 300), (64, 512, 2048), (130, 256, 100)])
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
