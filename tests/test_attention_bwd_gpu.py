"""The fused backward of fp32 attention on the torch device, against float64.

Sizes: one row, both sides of the 16-, 32- and 64-row edges of its tiles,
more keys than queries and fewer, every head dim it takes; q, k and v as views
of a fused projection, at offsets that are not 16-byte aligned, and expanded
gradients.  Bar: every product splits its operands into bf16 hi + lo (2^-16
per product, measured 8e-6 normwise after three chained products); 3e-5."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev(gpu):
    import torch
    from applegpu_runtime.cpp_backend import load_cpp_backend
    load_cpp_backend()
    return torch


def _reference(torch, q, k, v, go, causal, scale=None):
    q, k, v = (t.double().requires_grad_(True) for t in (q, k, v))
    s = q @ k.transpose(-1, -2) * (scale or q.shape[-1] ** -0.5)
    if causal:
        s = s.masked_fill(~torch.ones(s.shape[-2:], dtype=torch.bool).tril(), float("-inf"))
    out = torch.softmax(s, -1) @ v
    return (out.detach(),) + torch.autograd.grad(out, (q, k, v), go.double())


def _check(torch, got, want, names=("out", "dq", "dk", "dv"), bar=3e-5):
    for n, a, b in zip(names, got, want):
        a, b = a.detach().cpu().double(), b
        assert a.shape == b.shape and torch.isfinite(a).all(), n
        # a gradient that vanishes (one key: dS = P (dP - delta) = 0) is compared with the size of its
        # terms: dP of unit normals is sqrt(D) large, so a tenth of that bounds 2^-17 sqrt(D) by the bar
        ref = max(b.norm().item(), 0.1 * (b.shape[-1] * b.numel()) ** 0.5)
        assert (a - b).norm().item() <= bar * ref, (n, (a - b).norm().item() / ref)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Tq,Tk", [(1, 1), (1, 70), (15, 17), (16, 64), (63, 65), (64, 33), (65, 64), (130, 129),
                                   (257, 31), (40, 300)])
@pytest.mark.parametrize("causal", [False, True])
def test_gradients(torch_dev, Tq, Tk, D, causal):
    torch = torch_dev
    torch.manual_seed(Tq * 31 + Tk + D)
    q, go = torch.randn(2, 3, Tq, D), torch.randn(2, 3, Tq, D)
    k, v = torch.randn(2, 3, Tk, D), torch.randn(2, 3, Tk, D)
    dev = [t.to("applegpu").requires_grad_(True) for t in (q, k, v)]
    out = torch.nn.functional.scaled_dot_product_attention(*dev, is_causal=causal)
    got = (out,) + torch.autograd.grad(out, dev, go.to("applegpu"))
    _check(torch, got, _reference(torch, q, k, v, go, causal))


@pytest.mark.parametrize("offset", [0, 1, 4])
def test_views_of_a_projection(torch_dev, offset):
    """Heads of [B, T, 3 d] (strided, in place) at offsets that 16 bytes do
    and do not divide, and a gradient that is a transposed view."""
    torch = torch_dev
    B, T, H, D = 2, 77, 3, 64
    torch.manual_seed(offset)
    flat = torch.randn(offset + B * T * 3 * H * D)
    go = torch.randn(B, T, H, D)

    def heads(x):
        x = x[offset:].view(B, T, 3, H, D)
        return [x[:, :, j].transpose(1, 2) for j in range(3)]

    dev = flat.to("applegpu").requires_grad_(True)
    out = torch.nn.functional.scaled_dot_product_attention(*heads(dev), is_causal=True)
    (got,) = torch.autograd.grad(out, dev, go.to("applegpu").transpose(1, 2))
    q, k, v = heads(flat)
    want = _reference(torch, q, k, v, go.transpose(1, 2), True)
    ref = torch.cat([torch.zeros(offset).double(),
                     torch.stack([t.transpose(1, 2) for t in want[1:]], 2).reshape(-1)])
    _check(torch, (out, got), (want[0], ref), ("out", "dqkv"))


def test_partial_and_expanded_gradients(torch_dev):
    """Only some of q, k, v want a gradient; out.sum() gives a gradient of
    stride 0; 3-D operands; a scale of the caller's."""
    torch = torch_dev
    torch.manual_seed(9)
    q, k, v = (torch.randn(5, 50, 64) for _ in range(3))
    want = _reference(torch, q, k, v, torch.ones(5, 50, 64), False, 0.2)[1:]
    for wanted in ((0,), (1,), (2,), (0, 2)):
        dev = [t.to("applegpu").requires_grad_(i in wanted) for i, t in enumerate((q, k, v))]
        out = torch.nn.functional.scaled_dot_product_attention(*dev, scale=0.2)
        got = torch.autograd.grad(out.sum(), [dev[i] for i in wanted])
        _check(torch, got, [want[i] for i in wanted], wanted)


def test_same_bits_twice_and_rows_that_never_end(torch_dev):
    """Repeated calls agree bit for bit; large scores do not overflow; a NaN
    query makes its own gradient NaN and the others' keys and values too, as
    the products over the whole row do."""
    torch = torch_dev
    torch.manual_seed(10)
    q, k, v, go = (torch.randn(1, 4, 200, 64) for _ in range(4))
    q[0, 0] *= 40

    def grads(q):
        dev = [t.to("applegpu").requires_grad_(True) for t in (q, k, v)]
        out = torch.nn.functional.scaled_dot_product_attention(*dev, is_causal=True)
        return [t.cpu() for t in torch.autograd.grad(out, dev, go.to("applegpu"))]

    a, b = grads(q), grads(q)
    assert all(torch.equal(x, y) and torch.isfinite(x).all() for x, y in zip(a, b))
    q[0, 1, 7] = float("nan")
    c = grads(q)
    assert torch.isnan(c[0][0, 1, 7]).all() and torch.equal(c[0][0, 0], a[0][0, 0])
    assert torch.isnan(c[1][0, 1, 0]).all() and torch.equal(c[1][0, 2], a[1][0, 2])


def test_native_fp32_products(torch_dev):
    """With the native fp32 products chosen, the gradients keep their
    precision too (split products are 8e-6 off, fp32 sums of 300 terms 1e-6)."""
    torch = torch_dev
    from applegpu_runtime._native import lib
    torch.manual_seed(11)
    q, k, v, go = (torch.randn(2, 3, 300, 64) for _ in range(4))
    assert lib.applegpu_ffi_gemm_tune(1, -1, 0) == 0
    try:
        dev = [t.to("applegpu").requires_grad_(True) for t in (q, k, v)]
        out = torch.nn.functional.scaled_dot_product_attention(*dev, is_causal=True)
        got = (out,) + torch.autograd.grad(out, dev, go.to("applegpu"))
        _check(torch, got, _reference(torch, q, k, v, go, True), bar=1e-6)
    finally:
        lib.applegpu_ffi_gemm_tune(0, -1, 0)


@pytest.mark.parametrize("H,Tq,Tk,D,causal,fused", [
    (12, 128, 128, 64, True, True), (1, 16, 2048, 64, False, False), (1, 16, 2048, 64, True, True),
    (2, 2048, 16, 128, False, False), (1, 2048, 2048, 128, True, False), (12, 1024, 1024, 128, True, True),
    (1, 1023, 2049, 64, False, True), (3, 130, 4096, 32, False, False)])
def test_the_faster_way_is_taken(torch_dev, gpu, H, Tq, Tk, D, causal, fused):
    """A few heads with one long side take the products one by one: each of
    the fused kernels' blocks would walk that side alone."""
    torch = torch_dev
    torch.manual_seed(12)
    q, go = torch.randn(1, H, Tq, D), torch.randn(1, H, Tq, D)
    k, v = torch.randn(1, H, Tk, D), torch.randn(1, H, Tk, D)
    dev = [t.to("applegpu").requires_grad_(True) for t in (q, k, v)]
    out = torch.nn.functional.scaled_dot_product_attention(*dev, is_causal=causal)
    god = go.to("applegpu")
    before = gpu.graph_stats()["launcher_calls"]
    got = torch.autograd.grad(out, dev, god)
    assert (gpu.graph_stats()["launcher_calls"] - before <= 2) == fused
    _check(torch, (out,) + got, _reference(torch, q, k, v, go, causal))


def test_memory_limits_choose_the_way_that_fits(torch_dev, gpu):
    """One head of 2048 x 2048 takes the products over [2048, 2048] by itself,
    and the fused kernels where a limit leaves no room for those."""
    torch = torch_dev
    torch.manual_seed(13)
    q, k, v, go = (torch.randn(1, 1, 2048, 128) for _ in range(4))
    want = _reference(torch, q, k, v, go, False)
    dev = [t.to("applegpu").requires_grad_(True) for t in (q, k, v)]
    out = torch.nn.functional.scaled_dot_product_attention(*dev)
    god = go.to("applegpu")
    for limit, fused in ((dict(), False), (dict(max_tensor_size_mb=8), True),
                         (dict(max_memory_mb=(gpu.memory_usage() >> 20) + 24), True)):
        gpu.set_limits(**limit)
        try:
            before = gpu.graph_stats()["launcher_calls"]
            got = torch.autograd.grad(out, dev, god, retain_graph=True)
            assert (gpu.graph_stats()["launcher_calls"] - before <= 2) == fused
        finally:
            gpu.set_limits()
        _check(torch, (out,) + got, want)
        del got
