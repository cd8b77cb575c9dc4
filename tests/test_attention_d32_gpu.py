"""Fused attention at head dim 32 on the MFMA kernels, against float64: one
row, the edges of the 16-, 64- and 128-query blocks and the 64-key tiles,
fewer and more keys than queries, heads as views of a fused projection.
Bars: fp32 sums of at most Tk probabilities and 32 products, 2^-24 each,
averaging out to 1e-6 normwise; 16-bit results one rounding of the result
(2^-11, 2^-8 per element, half of that normwise), since the probabilities
keep more than 16 bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(32)
BAR = {"float32": 1e-6, "float16": 0.6 * 2.0 ** -11, "bfloat16": 0.6 * 2.0 ** -8}


def _want(q, k, v, causal):
    s = q @ np.swapaxes(k, -1, -2) / np.sqrt(32.0)
    if causal:
        s = np.where(np.tril(np.ones(s.shape[-2:], bool)), s, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    return (p / p.sum(-1, keepdims=True)) @ v


def _dev(gpu, a, dt):
    t = gpu.cast(gpu.from_numpy(a.astype(np.float32)), dt)
    return t, t.to_numpy().astype(np.float64)


@pytest.mark.parametrize("dt", list(BAR))
@pytest.mark.parametrize("B,H,Tq,Tk,causal", [(1, 1, 1, 1, True), (1, 2, 15, 70, False), (2, 3, 64, 64, True),
                                              (1, 3, 65, 63, True), (1, 2, 130, 200, True), (2, 40, 129, 257, False),
                                              (4, 70, 200, 200, True), (1, 5, 777, 777, True)])
def test_against_float64(gpu, dt, B, H, Tq, Tk, causal):
    (q, qs), (k, ks), (v, vs) = (_dev(gpu, RNG.standard_normal((B, H, t, 32)), dt) for t in (Tq, Tk, Tk))
    got = (gpu.attention_causal if causal else gpu.attention)(q, k, v).to_numpy().astype(np.float64)
    want = _want(qs, ks, vs, causal)
    assert np.linalg.norm(got - want) <= BAR[dt] * np.linalg.norm(want)


@pytest.mark.parametrize("dt", list(BAR))
def test_heads_of_a_projection(gpu, dt):
    """The head split and the head merge are views; with fp32 the merged heads
    may go straight into packed rows of the next product."""
    T, H, d = 100, 4, 128
    t, x = _dev(gpu, RNG.standard_normal((T, 3 * d)), dt)
    heads = [gpu.transpose_dims(gpu.reshape(gpu.slice(t, 1, j * d, (j + 1) * d), [T, H, 32]), 0, 1) for j in range(3)]
    hs = [x[:, j * d:(j + 1) * d].reshape(T, H, 32).transpose(1, 0, 2) for j in range(3)]
    want = _want(*hs, True).transpose(1, 0, 2).reshape(T, d)
    merged = gpu.reshape(gpu.transpose_dims(gpu.attention_causal(*heads), 0, 1), [T, d])
    got = merged.to_numpy().astype(np.float64)
    assert np.linalg.norm(got - want) <= BAR[dt] * np.linalg.norm(want)
    if dt == "float32":
        w, ws = _dev(gpu, RNG.standard_normal((d, 96)) * 0.1, dt)
        merged = gpu.reshape(gpu.transpose_dims(gpu.attention_causal(*heads), 0, 1), [T, d])
        y = gpu.matmul_pp(gpu.pack_rows_x3(merged), T, gpu.pack_weight_x3(w), 96).to_numpy().astype(np.float64)
        ref = want @ ws
        assert np.linalg.norm(y - ref) <= 1e-5 * np.linalg.norm(ref)   # the split products' 2^-17


@pytest.mark.parametrize("dt", list(BAR))
@pytest.mark.parametrize("B,H,Tq,Tk,causal", [(1, 1, 1, 1, True), (1, 2, 70, 70, True), (1, 2, 70, 130, False),
                                              (1, 2, 200, 200, True), (2, 70, 130, 130, True), (2, 70, 130, 90, False)])
def test_infinite_and_nan_values(gpu, dt, B, H, Tq, Tk, causal):
    """A key's infinite or NaN value reaches the queries that see the key, as
    itself, and no others: at the first and the last key, inside a tile and on
    the causal diagonal, beside finite ones in the same row."""
    a = RNG.standard_normal((B, H, Tk, 32))
    a[0, 0, 0, 3] = np.inf
    a[0, 0, Tk // 2, 5] = -np.inf
    a[0, 0, Tk // 3, 17] = np.nan
    a[0, 0, Tk - 1, 8:16] = np.inf
    a[-1, -1, Tk // 2, 30] = np.inf
    a[-1, -1, Tk - 1, 30] = -np.inf               # both signs: NaN where both are seen
    (q, qs), (k, ks) = (_dev(gpu, RNG.standard_normal((B, H, t, 32)), dt) for t in (Tq, Tk))
    v, vs = _dev(gpu, a, dt)
    got = (gpu.attention_causal if causal else gpu.attention)(q, k, v).to_numpy().astype(np.float64)
    want = np.empty((B, H, Tq, 32))
    see = np.tril(np.ones((Tq, Tk), bool)) if causal else np.ones((Tq, Tk), bool)
    s = np.where(see, qs @ np.swapaxes(ks, -1, -2) / np.sqrt(32.0), -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    with np.errstate(invalid="ignore"):
        for i in range(Tq):
            want[:, :, i] = (p[:, :, i, see[i], None] * vs[:, :, see[i]]).sum(2)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isposinf(got), np.isposinf(want))
    np.testing.assert_array_equal(np.isneginf(got), np.isneginf(want))
    ok = np.isfinite(want)
    assert np.linalg.norm(got[ok] - want[ok]) <= BAR[dt] * np.linalg.norm(want[ok])
