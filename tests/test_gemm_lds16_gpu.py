"""The direct-to-LDS 16-bit GEMM at the edges of its three tiles: rows and
columns one past and one short of a tile, a last stage of every length (K a
multiple of 8), a single stage, more tiles than one round of the CUs, odd
columns (rows of C at any alignment), every activation and a residual, and
operands that are row ranges of wider tensors; and products it declines.
Reference: float64 on the operands as stored; bar: the fp32 sum's rounding is
far below one rounding of the result (2^-11, 2^-8), with the residual's
rounding of a larger sum: 2 roundings of the largest term."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(77)
EPS = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}


def _plan(M, N, K, dt="float16"):
    from applegpu_runtime._native import lib
    buf = ctypes.create_string_buffer(96)
    assert lib.applegpu_ffi_gemm_plan(M, N, K, 1, {"float16": 1, "bfloat16": 10}[dt], True, True, buf, 96) == 0
    return buf.value.decode()


def _dev(gpu, a, dt):
    t = gpu.cast(gpu.from_numpy(np.ascontiguousarray(a, np.float32)), dt)
    return t, t.to_numpy().astype(np.float64)


def _close(got, ref, dt, size=0.0):
    bar = 2 * EPS[dt] * np.maximum(np.abs(ref), size) + 1e-4
    assert (np.abs(got.astype(np.float64) - ref) <= bar).all(), np.abs(got - ref).max()


@pytest.mark.parametrize("dt", ["float16", "bfloat16"])
@pytest.mark.parametrize("M,N,K,tile", [
    (1025, 1281, 64, "128x64"), (1151, 1345, 72, "128x64"), (2049, 1279, 136, "128x64"),
    (4000, 1023, 200, "128x64"), (1921, 3713, 1288, "128x128"), (1153, 5120, 1336, "128x128"),
    (300, 20001, 64, "128x128"), (4095, 3839, 72, "256x256"), (3000, 3841, 200, "256x256"),
    (2559, 5121, 1120, "256x256"),
])
def test_edges(gpu, M, N, K, tile, dt):
    plan = _plan(M, N, K, dt)
    assert plan.startswith("lds16") and tile in plan, plan
    (x, xs), (w, ws), (b, bs) = (_dev(gpu, RNG.standard_normal(s) * 0.3, dt) for s in ((M, K), (N, K), (N,)))
    got = gpu.linear(x, w, b).to_numpy()
    _close(got, xs @ ws.T + bs, dt)


@pytest.mark.parametrize("dt", ["float16", "bfloat16"])
@pytest.mark.parametrize("act", [None, "relu", "gelu", "gelu_exact"])
def test_epilogues(gpu, act, dt):
    from scipy.special import erf
    M, N, K = 1200, 1283, 88
    (x, xs), (w, ws), (b, bs), (r, rs) = (_dev(gpu, RNG.standard_normal(s) * 0.5, dt)
                                         for s in ((M, K), (N, K), (N,), (M, N)))
    z = xs @ ws.T + bs
    f = {None: z, "relu": np.maximum(z, 0), "gelu_exact": 0.5 * z * (1 + erf(z / np.sqrt(2))),
         "gelu": 0.5 * z * (1 + np.tanh(np.clip(0.7978845608 * (z + 0.044715 * z ** 3), -10, 10)))}[act]
    _close(gpu.linear(x, w, b, act).to_numpy(), f, dt)
    if act is None:
        got = (r + gpu.add_bias(x @ gpu.transpose(w), b)).to_numpy()
        _close(got, z + rs, dt, np.abs(z) + np.abs(rs))


def test_row_ranges_of_wider_tensors(gpu):
    M, N, K, ld = 1200, 1300, 104, 136
    (x, xs), (w, ws) = (_dev(gpu, RNG.standard_normal((n, ld)) * 0.5, "float16") for n in (M, N))
    for lo in (0, 8, 32, 3):   # 3: not 16-byte aligned, another plan
        xv, wv = gpu.slice(x, 1, lo, lo + K), gpu.slice(w, 1, lo, lo + K)
        got = (xv @ gpu.transpose(wv)).to_numpy()
        _close(got, xs[:, lo:lo + K] @ ws[:, lo:lo + K].T, "float16")


@pytest.mark.parametrize("both", [False, True])
def test_columns_of_a_tensor_past_2_gib(gpu, both):
    """A last stage of 8 k of rows 2 MiB apart: what lies 2 GiB behind a
    tile's first row, outside the columns multiplied, is not read as the
    stage's padding (an infinity there, or finite values on both sides)."""
    M, ld, K = 1100, 1 << 20, 72
    big = np.zeros((M, ld), np.float16)
    big[:, :2 * K] = RNG.standard_normal((M, 2 * K)) * 0.5
    big[1023, -8:] = 9.0 if both else np.inf     # byte 0x7ffffff0 from the tensor's first row
    x = gpu.from_numpy(big)
    xs = big[:, :2 * K].astype(np.float64)
    del big
    xv = gpu.slice(x, 1, 0, K)
    if both:
        wv, ws = gpu.slice(x, 1, K, 2 * K), xs[:, K:]
    else:
        wv, ws = _dev(gpu, RNG.standard_normal((M, K)) * 0.5, "float16")
    assert _plan(M, M, K).startswith("lds16")
    _close((xv @ gpu.transpose(wv)).to_numpy(), xs[:, :K] @ ws.T, "float16")


@pytest.mark.parametrize("dt", ["float16", "bfloat16"])
@pytest.mark.parametrize("M,N,K,here", [(17, 8192, 512, True), (64, 10240, 1024, True), (192, 5120, 1280, True),
                                        (17, 8192, 768, False), (64, 10240, 1280, False), (17, 10240, 2048, False),
                                        (192, 5120, 2048, False), (64, 16384, 2048, True)])
def test_few_rows_of_long_k_are_left_to_split_tiles(gpu, M, N, K, here, dt):
    assert _plan(M, N, K, dt).startswith("lds16" if here else "mf")
    (x, xs), (w, ws), (b, bs) = (_dev(gpu, RNG.standard_normal(s) * 0.1, dt) for s in ((M, K), (N, K), (N,)))
    _close(gpu.linear(x, w, b).to_numpy(), xs @ ws.T + bs, dt)


def test_declines():
    assert not _plan(1024, 1280, 100).startswith("lds16")    # rows of partial vectors
    assert not _plan(100, 1280, 1280).startswith("lds16")    # too few tiles
