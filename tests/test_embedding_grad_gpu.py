"""embedding and embedding_backward where their vector forms begin and end:
rows of whole and of partial vectors, buffers at odd offsets, words named
fewer times than the rows in flight, exactly as often, and by more tokens than
one gathering round holds.  Both are exact: the lookup copies, the gradient
adds rows in token order as the oracle does."""
import numpy as np
import pytest

from oracle import ops as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [1, 4, 5, 768, 1024, 1028, 2052])
@pytest.mark.parametrize("n", [1, 3, 16, 20, 63, 1025, 4500])
def test_gradient_of_one_hot_word(gpu, n, dim):
    rng = np.random.default_rng(n * 7 + dim)
    idx = rng.integers(0, 6, n).astype(np.int32)
    idx[rng.random(n) < 0.6] = 2   # one word beyond every list and unroll boundary
    idx[0] = -1 if n > 1 else 2
    dy = rng.standard_normal((n, dim)).astype(np.float32)
    got = gpu.embedding_backward(gpu.from_numpy(dy), gpu.from_numpy(idx), 9).to_numpy()
    np.testing.assert_array_equal(got, O.embedding_backward(dy, idx, 9))


@pytest.mark.parametrize("dt", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("lo,dim", [(0, 64), (1, 64), (2, 12), (3, 7)])
def test_odd_offsets(gpu, dt, lo, dim):
    """Tables and gradients that start inside a buffer, as a slice of rows of
    an odd-sized tensor does."""
    rng = np.random.default_rng(lo + dim)
    base = rng.standard_normal((lo + 50 * dim,)).astype(np.float32)
    t = gpu.from_numpy(base)
    if dt != "float32":
        t = gpu.cast(t, dt)
        base = t.to_numpy().astype(np.float32)
    part = gpu.reshape(gpu.slice(t, 0, lo, lo + 50 * dim), [50, dim])
    w = base[lo:].reshape(50, dim)
    idx = rng.integers(-2, 52, 37).astype(np.int64)
    ok = (idx >= 0) & (idx < 50)
    got = gpu.embedding(part, gpu.from_numpy(idx)).to_numpy().astype(np.float32)
    np.testing.assert_array_equal(got, np.where(ok[:, None], w[np.clip(idx, 0, 49)], 0))
    idx = rng.integers(0, 20, 50).astype(np.int64)
    got = gpu.embedding_backward(part, gpu.from_numpy(idx), 20).to_numpy().astype(np.float32)
    want = O.embedding_backward(w, idx, 20)
    if dt != "float32":
        want = gpu.cast(gpu.from_numpy(want.astype(np.float32)), dt).to_numpy().astype(np.float32)
    np.testing.assert_array_equal(got, want)
