"""Large fp16 / bf16 GEMMs with both operands contiguous along k (the C4
prefill's projections and LM head: x [M, K] @ W^T with W [N, K]) on the
swizzled direct-to-LDS tile kernel, whose largest tile fills one round of the
CUs here, against the float64 oracle on the
operands as stored, at the 16-bit bar (north star: 1e-2 fp16, 2e-2 bf16
relative), at the tile shape the plan picks, ragged edges and the fused
epilogues (bias, GELU, residual)."""
import ctypes

import numpy as np
import pytest

from conftest import rel_err
from oracle import ops as O

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(1607)
TOL = {"float16": 1e-2, "bfloat16": 2e-2}


def _plan(M, N, K, dt):
    from applegpu_runtime._native import lib
    buf = ctypes.create_string_buffer(96)
    assert lib.applegpu_ffi_gemm_plan(M, N, K, 1, {"float16": 1, "bfloat16": 10}[dt], True, True, buf, 96) == 0
    return buf.value.decode()


def _dev(gpu, a, dt):
    return gpu.cast(gpu.from_numpy(np.ascontiguousarray(a, np.float32)), dt)


def _stored(t):
    return np.asarray(t.to_numpy(), np.float64)


@pytest.mark.parametrize("dt", ["float16", "bfloat16"])
@pytest.mark.parametrize("M,N,K,tile", [(4096, 3840, 1280, "256x256"), (4000, 3900, 192, "256x256"),
                                        (4096, 3856, 64, "256x256"), (3072, 4608, 512, "256x256")])
def test_h16_tiles_vs_oracle(gpu, dt, M, N, K, tile):
    plan = _plan(M, N, K, dt)
    assert plan == "lds16 " + tile, plan
    x = _dev(gpu, RNG.standard_normal((M, K)), dt)
    w = _dev(gpu, RNG.standard_normal((N, K)) * 0.05, dt)
    got = np.asarray((x @ gpu.transpose(w)).to_numpy(), np.float32)
    ref = O.matmul(_stored(x), _stored(w).T)
    assert rel_err(got, ref) < TOL[dt]


@pytest.mark.parametrize("dt", ["float16", "bfloat16"])
def test_h16_fused_epilogues(gpu, dt):
    """Linear + bias + GELU, and Linear + bias + residual, each one launch."""
    M, N, K = 3072, 4096, 256
    assert _plan(M, N, K, dt) == "lds16 256x256"
    x = _dev(gpu, RNG.standard_normal((M, K)), dt)
    w = _dev(gpu, RNG.standard_normal((N, K)) * 0.05, dt)
    b = _dev(gpu, RNG.standard_normal(N), dt)
    r = _dev(gpu, RNG.standard_normal((M, N)), dt)
    for t in (x, w, b, r):
        t.eval()
    before = gpu.graph_stats()["launcher_calls"]
    y = gpu.gelu(gpu.add_bias(x @ gpu.transpose(w), b))
    z = r + gpu.add_bias(x @ gpu.transpose(w), b)
    got_y = np.asarray(y.to_numpy(), np.float32)
    got_z = np.asarray(z.to_numpy(), np.float32)
    assert gpu.graph_stats()["launcher_calls"] - before == 2
    lin = O.matmul(_stored(x), _stored(w).T) + _stored(b)
    assert rel_err(got_y, O.gelu_tanh(lin)) < TOL[dt]
    assert rel_err(got_z, lin + _stored(r)) < TOL[dt]


@pytest.mark.parametrize("M,N,K,tile", [(4096, 3840, 1280 + 32, "256x256"),   # a last stage of half its k
                                        (4096, 1280, 1280, "128x128"),        # 80 of the largest tiles
                                        (4096, 5120, 1280, "256x256"),        # 1.25 rounds of them
                                        (2000, 1280, 1280, "128x64")])
def test_h16_tile_of_other_grids(gpu, M, N, K, tile):
    assert _plan(M, N, K, "float16") == "lds16 " + tile
    x = _dev(gpu, RNG.standard_normal((M, K)), "float16")
    w = _dev(gpu, RNG.standard_normal((N, K)) * 0.05, "float16")
    got = np.asarray((x @ gpu.transpose(w)).to_numpy(), np.float32)
    assert rel_err(got, O.matmul(_stored(x), _stored(w).T)) < TOL["float16"]


def test_h16_declines():
    assert _plan(128, 3840, 1280, "float16").startswith("mf")        # few rows: fewer tiles than half the CUs
    assert _plan(4096, 3840, 1284, "float16").startswith("mf")       # rows that 16 bytes do not divide
    assert not _plan(8, 50257, 1280, "float16").startswith("lds16")  # the few-row kernel's
