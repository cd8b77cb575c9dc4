"""softmax, log_softmax, softmax_causal and layer_norm of long and unaligned
rows (16-byte vectors in registers) against float64.

Sizes: both sides of every change of wavefronts and vectors per thread, the
last size the registers hold and the first past it (of fp32 and of the 16-bit
types), rows that end inside a vector, and fewer rows than a block takes.  Bars: fp32 sums of at most 52
terms a thread, then a tree: 64 * 2^-24 = 4e-6 relative, log_softmax the same
absolute per unit of its magnitude; 16-bit results are one rounding of the
result (2^-11, 2^-8) plus the fp32 error."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COLS = [257, 300, 511, 513, 1023, 1025, 2047, 2049, 4096, 4099, 8192, 8193, 16385, 32769, 50257, 53248, 53249, 65536, 65537]
BAR = {"float32": 4e-6, "float16": 2.0 ** -11 + 4e-6, "bfloat16": 2.0 ** -8 + 4e-6}


def _rows(gpu, rows, cols, dt, seed=3):
    x = (np.random.default_rng(seed).standard_normal((rows, cols)) * 2).astype(np.float32)
    t = gpu.from_numpy(x)
    if dt != "float32":
        t = gpu.cast(t, dt)
        x = t.to_numpy().astype(np.float32)
    return t, x.astype(np.float64)


def _softmax64(x):
    e = np.exp(x - x.max(-1, keepdims=True))
    return e / e.sum(-1, keepdims=True)


@pytest.mark.parametrize("dt", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("cols", COLS)
def test_softmax_and_layer_norm(gpu, cols, dt):
    rows = 5 if cols < 3000 else 3
    t, x = _rows(gpu, rows, cols, dt)
    bar = BAR[dt]
    tiny = 2.0 ** -24 if dt == "float16" else 0.0   # half of float16's smallest step
    p = _softmax64(x)
    np.testing.assert_allclose(gpu.softmax(t).to_numpy().astype(np.float64), p, rtol=bar, atol=tiny)
    np.testing.assert_allclose(gpu.log_softmax(t).to_numpy().astype(np.float64), np.log(p), rtol=bar, atol=4e-6)
    g, gx = _rows(gpu, 1, cols, dt, 4)
    b, bx = _rows(gpu, 1, cols, dt, 5)
    got = gpu.layer_norm(t, gpu.reshape(g, [cols]), gpu.reshape(b, [cols])).to_numpy().astype(np.float64)
    n = (x - x.mean(-1, keepdims=True)) / np.sqrt(x.var(-1, keepdims=True) + 1e-5)
    # the sum with beta cancels: absolute bar at the largest term's size
    np.testing.assert_allclose(got, gx * n + bx, rtol=bar, atol=4e-6 * np.abs(gx * n).max())


@pytest.mark.parametrize("cols", [259, 1000, 2500, 9001])
def test_causal_masked_and_extreme_rows(gpu, cols):
    """Causal rows, -inf columns (a mask of the type's lowest value keeps its
    own meaning), +inf and NaN rows, the values at the row's two ends."""
    t, x = _rows(gpu, cols, cols, "float32")
    want = np.stack([np.r_[_softmax64(x[i:i + 1, :i + 1])[0], np.zeros(cols - i - 1)] for i in (0, 1, cols - 2, cols - 1)])
    got = gpu.softmax_causal(t).to_numpy().astype(np.float64)
    np.testing.assert_allclose(got[[0, 1, cols - 2, cols - 1]], want, rtol=4e-6, atol=0)
    assert (np.triu(got, 1) == 0).all()
    x = x[:6].astype(np.float32)
    x[0, 1:] = -np.inf                              # one column left, the first
    x[1, :-1] = np.finfo(np.float32).min            # the last, beside the lowest value
    x[2, :] = -np.inf
    x[3, cols // 2] = np.nan
    x[4, -1] = np.inf
    got = gpu.softmax(gpu.from_numpy(x)).to_numpy()
    assert got[0, 0] == 1 and (got[0, 1:] == 0).all()
    assert got[1, -1] == 1 and (got[1, :-1] == 0).all()
    assert np.isnan(got[2]).all() and np.isnan(got[3]).all() and np.isnan(got[4]).all()
    np.testing.assert_allclose(got[5], _softmax64(x[5:6].astype(np.float64))[0], rtol=4e-6, atol=0)


def test_rows_of_a_wider_tensor(gpu):
    """Rows whose stride is not their length, at an offset that only the
    elements' own size divides."""
    t, x = _rows(gpu, 7, 1203, "float32")
    for lo, hi in ((1, 1000), (3, 1203)):
        got = gpu.softmax(gpu.slice(t, 1, lo, hi)).to_numpy().astype(np.float64)
        np.testing.assert_allclose(got, _softmax64(x[:, lo:hi]), rtol=4e-6, atol=0)


@pytest.mark.parametrize("dt", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("cols", [64, 300, 512, 2048, 2500, 4099, 16385, 53249, 65537])
def test_rows_of_large_magnitude(gpu, cols, dt):
    """Rows of one value (every column masked with the type's lowest value, or
    with -1e9 or -1e10, and large positive ones), rows half masked, and rows
    far from zero whose columns differ: the exponents come from differences
    with the maximum, which are as exact there as around zero."""
    t, x = _rows(gpu, 10, cols, dt, 7)
    x = x.astype(np.float32)
    lowest = {"float32": -3.4028234e38, "float16": -65504.0, "bfloat16": -3.3895314e38}[dt]
    for r, v in enumerate((lowest, -1e9, -1e10, -1e12, 1e6, -lowest)):
        x[r] = np.clip(v, lowest, -lowest)
    x[6, ::2] = lowest
    x[7, :-1] = lowest
    x[8] = np.round(x[8]) * 256 + 32768.0        # steps of 256: 16-bit values too
    x[9] = np.round(x[9]) * 256 - 32768.0
    t = gpu.cast(gpu.from_numpy(x), dt) if dt != "float32" else gpu.from_numpy(x)
    x = t.to_numpy().astype(np.float64)
    p = _softmax64(x)
    e = x - x.max(-1, keepdims=True)
    log_p = e - np.log(np.exp(e).sum(-1, keepdims=True))
    tiny = 2.0 ** -24 if dt == "float16" else 2.0 ** -126   # below the smallest normal value
    np.testing.assert_allclose(gpu.softmax(t).to_numpy().astype(np.float64), p, rtol=BAR[dt], atol=tiny)
    got = gpu.log_softmax(t).to_numpy().astype(np.float64)
    # a log-probability near the type's lowest value may be its infinity
    far = log_p < lowest * (1 - 2.0 ** -9)
    assert (got[far] <= lowest * (1 - 2.0 ** -9)).all()
    np.testing.assert_allclose(got[~far], log_p[~far], rtol=BAR[dt], atol=4e-6)
    causal = gpu.softmax_causal(t).to_numpy().astype(np.float64)     # row r: its first r + 1 columns
    for r in range(10):
        want = np.r_[_softmax64(x[r:r + 1, :r + 1])[0], np.zeros(cols - r - 1)]
        np.testing.assert_allclose(causal[r], want, rtol=BAR[dt], atol=tiny)
