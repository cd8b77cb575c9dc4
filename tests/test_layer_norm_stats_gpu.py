"""layer_norm's row statistics on the torch device come from the launch that
normalises: mean and 1/sqrt(var + eps) against float64 for each kernel that
can write them (short rows, aligned rows of whole 256 columns, rows in
registers at odd lengths, rows past them), each type, strided rows, and the
gradients that they lead to.

Bars: the normalised rows and the statistics are fp32 sums rounded once to
the type; of values of order 1, 2^-22 absolute in fp32 (a few roundings of a
sum over the row divided by its length), one unit of the type otherwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev(gpu):
    import torch
    from applegpu_runtime.cpp_backend import load_cpp_backend
    load_cpp_backend()
    return torch


@pytest.mark.parametrize("dt", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("shape", [(1, 1), (7,), (5, 255), (3, 4, 256), (9, 777), (2, 2048), (3, 5000), (2, 60001),
                                   (0, 64)])
def test_statistics(torch_dev, dt, shape):
    torch = torch_dev
    dtype = getattr(torch, dt)
    gen = torch.Generator().manual_seed(sum(shape))
    x = (torch.randn(shape, generator=gen) * 2 + 0.5).to(dtype)
    C = shape[-1]
    g, b = torch.randn(C, generator=gen).to(dtype), torch.randn(C, generator=gen).to(dtype)
    eps = 1e-3
    y, mean, rstd = torch.native_layer_norm(x.to("applegpu"), (C,), g.to("applegpu"), b.to("applegpu"), eps)
    xd = x.double()
    m = xd.mean(-1, keepdim=True)
    r = 1.0 / torch.sqrt(((xd - m) ** 2).mean(-1, keepdim=True) + eps)
    want = (xd - m) * r * g.double() + b.double()
    assert y.shape == x.shape and mean.shape == m.shape and rstd.shape == m.shape
    assert y.dtype == mean.dtype == rstd.dtype == dtype
    u = {"float32": 2.0 ** -21, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}[dt]
    for got, ref in ((y, want), (mean, m), (rstd, r)):
        err = (got.cpu().double() - ref).abs()
        # one rounding of the type beside the fp32 error, which a large rstd
        # (a row of one column: 1/sqrt(eps)) scales
        assert bool((err <= u * (1.0 + ref.abs()) + 2.0 ** -21 * r.abs() * (1.0 + g.abs().max().double() * (1.0 + m.abs()))
                     if ref.shape == want.shape else err <= u * (1.0 + ref.abs())).all())


def test_strided_rows_and_gradients(torch_dev):
    torch = torch_dev
    import torch.nn.functional as F
    gen = torch.Generator().manual_seed(3)
    x0 = torch.randn(6, 10, 200, generator=gen)
    g0, b0 = torch.randn(96, generator=gen), torch.randn(96, generator=gen)
    go = torch.randn(10, 6, 96, generator=gen)

    def run(dev, dt):
        x, g, b = (t.to(dt).to(dev).requires_grad_() for t in (x0, g0, b0))
        y = F.layer_norm(x.transpose(0, 1)[..., 7:103], (96,), g, b, 1e-5)
        y.backward(go.to(dt).to(dev))
        return [t.detach().cpu().double() for t in (y, x.grad, g.grad, b.grad)]

    for got, want in zip(run("applegpu", torch.float32), run("cpu", torch.float64)):
        assert float((got - want).norm()) <= 2e-6 * float(want.norm())
