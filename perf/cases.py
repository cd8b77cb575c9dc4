"""The work that users of the framework have it do, as cases that can be timed
and compared: training steps of MLPs, GPT-2 forwards, prefills and decode
steps, the training of a transformer block on the torch device, and the single
layers that these are made of (linear, attention, int8 layers, row and
embedding ops), each through the public entry points.

`listed()` gives the fixed cases, `draw(rng)` one more of the same ranges;
`prepare`, `run`, `work`, `tolerance` and `exact` take a case.  Inputs are made
on the GPU from the seed; `exact` computes the same outputs in float64 with
plain torch.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "applegpu-runtime_amd"))

import applegpu_runtime as gpu  # noqa: E402
from applegpu_runtime import eager as E  # noqa: E402
from applegpu_runtime._native import lib  # noqa: E402
from applegpu_runtime.cpp_backend import load_cpp_backend  # noqa: E402
from applegpu_runtime.models import gpt2 as G  # noqa: E402
from applegpu_runtime.models.mlp import EagerMLP  # noqa: E402

VOCAB = 50257
SIZE = {"float32": 4, "float16": 2, "bfloat16": 2}
LR = 0.01


# ── the cases ───────────────────────────────────────────────────────────────
def listed():
    return [
        # the smallest training step: a two-layer net at a batch of 32, where
        # only the latency of a call counts
        dict(name="mlp_step_small", kind="mlp_step", d_in=64, hidden=128, d_out=10, layers=2, batch=32),
        # the headline's training step: two 4096-wide hidden layers, batch 256
        dict(name="mlp_step_wide", kind="mlp_step", d_in=4096, hidden=4096, d_out=1, layers=3, batch=256),
        # the headline's forward: GPT-2 small in fp32 over one sequence of 128
        dict(name="gpt2_forward_f32", kind="gpt2_forward", model="gpt2", n_layer=12, T=128),
        # the prompts of a batch in fp16 (layers of GPT-2 large with its head),
        # at a length that no tile divides
        dict(name="gpt2_prefill_f16", kind="gpt2_prefill", model="gpt2-large", n_layer=4, B=4, T=500,
             dtype="float16"),
        # one token for each of 8 sequences against their KV caches
        dict(name="gpt2_decode_f16", kind="gpt2_decode", model="gpt2-large", n_layer=4, B=8, context=600,
             dtype="float16"),
        # forward and backward of one GPT-2 small block under torch autograd on
        # the applegpu device: what a training step spends its time on
        dict(name="block_train_f32", kind="block_train", d=768, B=4, T=512),
        # attention alone, forward and backward, on the torch device, at a
        # ragged length
        dict(name="attention_train_f32", kind="attention_train", B=2, H=12, T=777, D=64, causal=True),
        # attention alone, forward, for long prompts in bf16
        dict(name="attention_bf16", kind="attention", B=2, H=20, T=1000, D=64, causal=True, dtype="bfloat16"),
        # a transformer's widening layer in bf16 at a ragged row count
        dict(name="linear_gelu_bf16", kind="linear", M=1111, K=1280, N=5120, act="gelu", dtype="bfloat16"),
        # an int8 layer for a few rows of fp32 activations
        dict(name="linear_int8", kind="linear_int8", M=64, K=8192, N=8192),
        # the row op over the vocabulary that the loss of a language model starts with
        dict(name="log_softmax_vocab", kind="rows", op="log_softmax", rows=2047, cols=VOCAB, dtype="float32"),
        # the token embedding of a training step, lookup and gradient, words as
        # frequent as in a text
        dict(name="embedding_train", kind="embedding_train", tokens=4096, vocab=VOCAB, d=768),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["mlp_step", "gpt2_forward", "gpt2_prefill", "gpt2_decode", "block_train", "attention_train",
                       "attention", "linear", "linear_int8", "rows", "embedding_train", "quantize"])
    half = rng.choice(["float16", "bfloat16"])
    if kind == "mlp_step":
        return dict(kind=kind, d_in=_log(rng, 8, 4096), hidden=_log(rng, 16, 4096), d_out=rng.randint(1, 10),
                    layers=rng.randint(2, 3), batch=_log(rng, 4, 256))
    if kind == "gpt2_forward":
        return dict(kind=kind, model=rng.choice(["gpt2", "gpt2-medium"]), n_layer=rng.randint(1, 6),
                    T=_log(rng, 4, 1024))
    if kind == "gpt2_prefill":
        B = _log(rng, 1, 8)
        return dict(kind=kind, model=rng.choice(["gpt2", "gpt2-medium", "gpt2-large"]), n_layer=rng.randint(1, 4),
                    B=B, T=_log(rng, 16, min(1024, 2000 // B)), dtype=half)
    if kind == "gpt2_decode":
        return dict(kind=kind, model=rng.choice(["gpt2", "gpt2-medium", "gpt2-large"]), n_layer=rng.randint(1, 4),
                    B=_log(rng, 1, 16), context=_log(rng, 16, 1023), dtype=half)
    if kind == "block_train":
        B = _log(rng, 1, 8)
        return dict(kind=kind, d=64 * rng.randint(4, 16), B=B, T=_log(rng, 16, min(1024, 4096 // B)))
    if kind == "attention_train":
        B = _log(rng, 1, 4)
        return dict(kind=kind, B=B, H=rng.randint(4, 16), T=_log(rng, 16, 1024), D=rng.choice([32, 64, 64, 128]),
                    causal=rng.random() < 0.75)
    if kind == "attention":
        return dict(kind=kind, B=_log(rng, 1, 8), H=rng.randint(4, 20), T=_log(rng, 16, 2048),
                    D=rng.choice([32, 64, 64, 128]), causal=rng.random() < 0.75,
                    dtype=rng.choice(["float32", half, half]))
    if kind == "linear":
        return dict(kind=kind, M=_log(rng, 1, 4096), K=_log(rng, 64, 5120), N=_log(rng, 64, 5120),
                    act=rng.choice(["", "relu", "gelu"]), dtype=rng.choice(["float32", half]))
    if kind == "linear_int8":
        return dict(kind=kind, M=_log(rng, 1, 256), K=_log(rng, 256, 8192), N=_log(rng, 256, 8192))
    if kind == "rows":
        rows = _log(rng, 16, 8192)
        return dict(kind=kind, op=rng.choice(["softmax", "log_softmax", "layer_norm"]), rows=rows,
                    cols=_log(rng, 64, min(VOCAB, 100_000_000 // rows)), dtype=rng.choice(["float32", half]))
    if kind == "quantize":
        return dict(kind=kind, rows=_log(rng, 64, 8192), cols=_log(rng, 64, 8192))
    return dict(kind=kind, tokens=_log(rng, 16, 8192), vocab=_log(rng, 1000, VOCAB), d=64 * rng.randint(4, 20))


# ── between torch's GPU tensors and the framework's ─────────────────────────
class _Buffer:
    """A device buffer as torch takes one; keeps its owner alive."""

    def __init__(self, ptr, shape, strides, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "strides": tuple(strides), "typestr": typestr,
                                         "data": (int(ptr), False), "version": 3}


_TYPESTR = {"float32": "<f4", "float16": "<f2", "bfloat16": "<i2", "int32": "<i4", "int8": "|i1"}


def _seen(ptr, shape, strides, dtype, owner):
    """The buffer at ptr as a torch tensor, in place (strides in elements)."""
    code = _TYPESTR[dtype]
    size = int(code[-1])
    t = torch.as_tensor(_Buffer(ptr, shape, [s * size for s in strides], code, owner), device="cuda")
    return t.view(torch.bfloat16) if dtype == "bfloat16" else t


def _view(t):
    """A GpuTensor's or EagerTensor's values as a torch tensor, in place."""
    if isinstance(t, gpu.GpuTensor):
        return _seen(lib.applegpu_eager_data_ptr(t.id), t.shape, t.strides(), t.dtype, t)
    shape = t.shape
    strides = [math.prod(shape[i + 1:]) for i in range(len(shape))]
    return _seen(lib.applegpu_eager_data_ptr(t.id), shape, strides, t.dtype, t)


def _back(t):
    """A tensor of the applegpu torch device as one of torch's GPU, in place."""
    return _seen(t.data_ptr(), t.shape, t.stride(), str(t.dtype).replace("torch.", ""), t)


def _upload(t):
    """A GpuTensor with the values of a contiguous tensor on torch's GPU."""
    out = gpu.zeros(list(t.shape), str(t.dtype).replace("torch.", ""))
    gpu.synchronize()
    _view(out).copy_(t)
    torch.cuda.synchronize()
    return out


def _rand(seed):
    g = torch.Generator("cuda")
    g.manual_seed(int(seed))

    def randn(*shape, std=1.0, mean=0.0, dtype="float32"):
        x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
        return (x * std + mean).to(getattr(torch, dtype))

    return g, randn


def _words(g, shape, vocab):
    """Token ids whose frequency falls with their rank, as words in a text."""
    u = torch.rand(shape, generator=g, device="cuda", dtype=torch.float64)
    return (torch.exp(u * math.log(vocab + 1.0)) - 1.0).floor().clamp_(0, vocab - 1).to(torch.int32)


# ── inputs, from the seed alone ─────────────────────────────────────────────
def _config(c):
    return dict(G.GPT2_CONFIGS[c["model"]], n_layer=c["n_layer"])


def _gpt2_weights(cfg, randn):
    """GPT-2's weights as fp32 tensors: matrices N(0, 0.02), small biases,
    layer-norm scales around 1."""
    out = {}
    for name, shape in G.weight_shapes(cfg).items():
        if name.endswith(".bias"):
            out[name] = randn(*shape, std=0.02)
        elif ".ln_" in name:
            out[name] = randn(*shape, std=0.1, mean=1.0)
        else:
            out[name] = randn(*shape, std=0.02)
    return out


def _sizes(c):
    return [c["d_in"]] + [c["hidden"]] * (c["layers"] - 1) + [c["d_out"]]


BLOCK = ("g1", "b1", "wqkv", "bqkv", "wo", "bo", "g2", "b2", "wfc", "bfc", "wproj", "bproj")


def _inputs(c, seed):
    """The case's input tensors on torch's GPU, as the path is given them."""
    g, randn = _rand(seed)
    kind = c["kind"]
    if kind == "mlp_step":
        sizes, params = _sizes(c), []
        for fin, fout in zip(sizes[:-1], sizes[1:]):   # torch.nn.Linear's own initialisation
            bound = 1.0 / math.sqrt(fin)
            w = (torch.rand((fout, fin), generator=g, device="cuda") * 2 - 1) * bound
            b = (torch.rand((fout,), generator=g, device="cuda") * 2 - 1) * bound
            params.append((w, b))
        return dict(params=params, x=randn(c["batch"], c["d_in"]), y=randn(c["batch"], c["d_out"]))
    if kind in ("gpt2_forward", "gpt2_prefill", "gpt2_decode"):
        cfg = _config(c)
        d = dict(weights=_gpt2_weights(cfg, randn))
        if kind == "gpt2_forward":
            return dict(d, ids=_words(g, (1, c["T"]), VOCAB))
        if kind == "gpt2_prefill":
            return dict(d, ids=_words(g, (c["B"], c["T"]), VOCAB))
        shape = (c["B"], cfg["n_head"], c["context"], cfg["n_embd"] // cfg["n_head"])
        kv = [randn(*shape, std=0.7, dtype=c["dtype"]) for _ in range(2 * cfg["n_layer"])]
        return dict(d, ids=_words(g, (c["B"],), VOCAB), k=kv[0::2], v=kv[1::2])
    if kind == "block_train":
        d = c["d"]
        shapes = dict(g1=(d,), b1=(d,), wqkv=(3 * d, d), bqkv=(3 * d,), wo=(d, d), bo=(d,), g2=(d,), b2=(d,),
                      wfc=(4 * d, d), bfc=(4 * d,), wproj=(d, 4 * d), bproj=(d,))
        p = {k: randn(*s, std=0.1, mean=1.0) if k in ("g1", "g2") else randn(*s, std=0.02 if len(s) == 1 else 0.04)
             for k, s in shapes.items()}
        return dict(p, x=randn(c["B"], c["T"], d), go=randn(c["B"], c["T"], d, std=1e-2))
    if kind == "attention_train":
        shape = (c["B"], c["H"], c["T"], c["D"])
        return dict(q=randn(*shape), k=randn(*shape), v=randn(*shape), go=randn(*shape))
    if kind == "attention":
        shape = (c["B"], c["H"], c["T"], c["D"])
        return {k: randn(*shape, dtype=c["dtype"]) for k in ("q", "k", "v")}
    if kind == "linear":
        dt = c["dtype"]
        return dict(x=randn(c["M"], c["K"], dtype=dt), w=randn(c["N"], c["K"], std=1 / math.sqrt(c["K"]), dtype=dt),
                    b=randn(c["N"], std=0.1, dtype=dt))
    if kind == "linear_int8":
        return dict(x=randn(c["M"], c["K"]), w=randn(c["N"], c["K"], std=0.02))
    if kind == "quantize":
        return dict(w=randn(c["rows"], c["cols"], std=0.02))
    if kind == "rows":
        dt = c["dtype"]
        return dict(x=randn(c["rows"], c["cols"], std=2.0, dtype=dt), g=randn(c["cols"], std=0.1, mean=1.0, dtype=dt),
                    b=randn(c["cols"], std=0.1, dtype=dt))
    return dict(ids=_words(g, (c["tokens"],), c["vocab"]), w=randn(c["vocab"], c["d"], std=0.02),
                go=randn(c["tokens"], c["d"], std=1e-2))


# ── what a user's program has in hand, and one pass ─────────────────────────
def _captured(fn, *tensors):
    """The program records its layer once as a graph, over inputs that stay
    on the device, and replays it."""
    graph = gpu.capture(fn)
    out = graph.outputs if isinstance(graph.outputs, (list, tuple)) else [graph.outputs]
    return dict(run="replay", graph=graph, inputs=tensors, out=[_view(t) for t in out])


def prepare(case, seed):
    c, kind = case, case["kind"]
    gpu.init_backend()
    i = _inputs(c, seed)
    if kind == "mlp_step":
        mlp = EagerMLP([(w.cpu().numpy(), b.cpu().numpy()) for w, b in i["params"]])
        out = [_view(t) for p in mlp.params for t in p]
        return dict(run="mlp_step", mlp=mlp, x=E.from_numpy(i["x"].cpu().numpy()), y=E.from_numpy(i["y"].cpu().numpy()),
                    out=out)
    if kind in ("gpt2_forward", "gpt2_prefill", "gpt2_decode"):
        cfg = _config(c)
        model = G.load_model({k: w.cpu().numpy() for k, w in i["weights"].items()}, cfg, c.get("dtype", "float32"))
        if kind == "gpt2_forward":
            ids = _upload(i["ids"][0])
            pos = gpu.from_numpy(np.arange(c["T"], dtype=np.int32))
            return _captured(lambda: G.gpt2_forward(model, ids, positions=pos, need_cache=False)[0], model, ids, pos)
        if kind == "gpt2_prefill":
            gen = G.Generation(model, i["ids"].cpu().numpy(), 0)
            out = [_view(gen.graphs[0].outputs)] + [_view(t) for t in gen.cache.k + gen.cache.v]
            return dict(run="gpt2_prefill", gen=gen, out=out)
        cache = G.KVCache(cfg, c["B"], c["context"] + 1, c["dtype"])
        gpu.synchronize()
        for t, rows in zip(cache.k + cache.v, i["k"] + i["v"]):
            _view(t)[:, :, :c["context"]].copy_(rows)
        torch.cuda.synchronize()
        cache.pos.write(np.full(c["B"], c["context"], np.int32))
        tokens = _upload(i["ids"])
        s = _captured(lambda: G.gpt2_decode_step(model, tokens, cache)[0], model, tokens, cache)
        s["out"] += [_view(t)[:, :, c["context"]] for t in cache.k + cache.v]   # the rows that the step appends
        return s
    if kind in ("block_train", "attention_train"):
        load_cpp_backend()
        t = {k: v.cpu().to("applegpu") for k, v in i.items()}
        for k in t:
            if k != "go":
                t[k].requires_grad_(True)
        return dict(run=kind, case=dict(c), **t)
    t = {k: _upload(v) for k, v in i.items()}
    if kind == "attention":
        op = gpu.attention_causal if c["causal"] else gpu.attention
        return _captured(lambda: op(t["q"], t["k"], t["v"]), t)
    if kind == "linear":
        return _captured(lambda: gpu.linear(t["x"], t["w"], t["b"], c["act"] or None), t)
    if kind == "linear_int8":
        q, scale = gpu.quantize_per_row(t["w"])
        gpu.eval_many([q, scale])
        return _captured(lambda: gpu.linear_int8(t["x"], q, scale), t, q, scale)
    if kind == "quantize":
        def both():
            q, scale = gpu.quantize_per_row(t["w"])
            return q, scale, gpu.dequantize_per_row(q, scale)
        return _captured(both, t)
    if kind == "rows":
        if c["op"] == "layer_norm":
            return _captured(lambda: gpu.layer_norm(t["x"], t["g"], t["b"]), t)
        return _captured(lambda: (gpu.softmax if c["op"] == "softmax" else gpu.log_softmax)(t["x"]), t)
    return _captured(lambda: (gpu.embedding(t["w"], t["ids"]), gpu.embedding_backward(t["go"], t["ids"], c["vocab"])), t)


def _block(s, c, d_head=64):
    """One pre-norm GPT-2 block on x [B, T, d]."""
    B, T, d = c["B"], c["T"], c["d"]
    H = d // d_head
    x = s["x"].view(B * T, d)
    h = F.layer_norm(x, (d,), s["g1"], s["b1"])
    qkv = F.linear(h, s["wqkv"], s["bqkv"]).view(B, T, 3, H, d_head)
    q, k, v = (qkv[:, :, j].transpose(1, 2) for j in range(3))
    a = F.scaled_dot_product_attention(q, k, v, is_causal=True)
    x = x + F.linear(a.transpose(1, 2).reshape(B * T, d), s["wo"], s["bo"])
    h = F.layer_norm(x, (d,), s["g2"], s["b2"])
    f = F.gelu(F.linear(h, s["wfc"], s["bfc"]), approximate="tanh")
    return (x + F.linear(f, s["wproj"], s["bproj"])).view(B, T, d)


def run(state):
    s = state
    if s["run"] == "replay":
        s["graph"].replay()
        return s["out"]
    if s["run"] == "gpt2_prefill":
        s["gen"].prefill()
        return s["out"]
    if s["run"] == "mlp_step":
        loss = s["mlp"].train_step(s["x"], s["y"], LR)
        return [_view(loss)] + s["out"]
    if s["run"] == "block_train":
        out = _block(s, s["case"])
        grads = torch.autograd.grad(out, [s[k] for k in ("x",) + BLOCK], s["go"])
    else:
        out = F.scaled_dot_product_attention(s["q"], s["k"], s["v"], is_causal=s["case"]["causal"])
        grads = torch.autograd.grad(out, [s["q"], s["k"], s["v"]], s["go"])
    return [_back(t) for t in (out.detach(),) + grads]


# ── what a pass cannot do without ───────────────────────────────────────────
def work(case):
    c, kind = case, case["kind"]
    if kind == "mlp_step":
        sizes, B = _sizes(c), c["batch"]
        n = sum(a * b for a, b in zip(sizes[:-1], sizes[1:]))
        # forward, dW of each layer, dX of each but the first; parameters read and written
        return dict(bytes=4 * (2 * (n + sum(sizes[1:])) + B * (sizes[0] + sizes[-1])),
                    flops=2 * B * (3 * n - sizes[0] * sizes[1]))
    if kind in ("gpt2_forward", "gpt2_prefill", "gpt2_decode"):
        cfg = _config(c)
        d, L, e = cfg["n_embd"], c["n_layer"], SIZE[c.get("dtype", "float32")]
        B = c.get("B", 1)
        n = B if kind == "gpt2_decode" else B * c["T"]
        weights = L * 12 * d * d + VOCAB * d
        kv = 2 * L * d * (B * (c["context"] + 1) if kind == "gpt2_decode" else n if kind == "gpt2_prefill" else 0)
        pairs = B * (c["context"] + 1) if kind == "gpt2_decode" else B * c["T"] * (c["T"] + 1) / 2
        return dict(bytes=e * (weights + kv + n * VOCAB), flops=2 * n * weights + 4 * L * d * pairs)
    if kind == "block_train":
        d, n = c["d"], c["B"] * c["T"]
        pairs = c["B"] * c["T"] * (c["T"] + 1) / 2
        # attention forward: 2 products over the pairs; backward: 5
        return dict(bytes=4 * (2 * 12 * d * d + 4 * n * d), flops=3 * 2 * n * 12 * d * d + 7 * 2 * d * pairs)
    if kind in ("attention", "attention_train"):
        n = c["B"] * c["H"] * c["T"] * c["D"]
        pairs = c["B"] * c["H"] * c["T"] * ((c["T"] + 1) / 2 if c["causal"] else c["T"])
        if kind == "attention":
            return dict(bytes=4 * n * SIZE[c["dtype"]], flops=4 * c["D"] * pairs)
        return dict(bytes=8 * n * 4, flops=14 * c["D"] * pairs)
    if kind == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        return dict(bytes=SIZE[c["dtype"]] * (M * K + K * N + N + M * N), flops=2 * M * K * N)
    if kind == "linear_int8":
        M, K, N = c["M"], c["K"], c["N"]
        return dict(bytes=4 * M * K + K * N + 4 * N + 4 * M * N, flops=2 * M * K * N)
    if kind == "quantize":
        n = c["rows"] * c["cols"]
        return dict(bytes=9 * n + 4 * c["rows"], flops=4 * n)
    if kind == "rows":
        n = c["rows"] * c["cols"]
        return dict(bytes=2 * SIZE[c["dtype"]] * n, flops=5 * n)
    n = c["tokens"] * c["d"]
    return dict(bytes=4 * (3 * n + c["vocab"] * c["d"]), flops=n)


def tolerance(case):
    """About four times the measured distance from `exact` (in brackets)."""
    c, kind = case, case["kind"]
    half = c.get("dtype", "float32") != "float32"
    bf16 = c.get("dtype") == "bfloat16"
    if kind == "quantize":   # codes differ only where a value lies on a rounding boundary
        return dict(rel=1e-6, max=1e-2, differ=1e-5)
    if kind == "embedding_train":   # [2.2e-7]
        return dict(rel=1e-6, max=1e-4)
    if kind == "mlp_step":   # [1.4e-6 at the widest, weights and their update together]
        return dict(rel=1e-5, max=1e-3)
    if kind in ("gpt2_forward", "gpt2_prefill", "gpt2_decode"):   # [1.3e-5, f16 8.5e-4, bf16 eight times that]
        return dict(rel=2.5e-2 if bf16 else 4e-3, max=0.3) if half else dict(rel=5e-5, max=2e-3)
    if half:   # [2.0e-3 in bf16, 2.1e-4 in f16: one rounding of the result]
        return dict(rel=8e-3 if bf16 else 1e-3, max=0.1)
    if kind == "rows":   # [4e-8 to 2e-7]
        return dict(rel=1e-6, max=1e-4)
    return dict(rel=5e-5, max=2e-3)   # [3e-7 to 1.4e-5: products of fp32 values split into bf16 pairs]


# ── the same outputs in 64 bits, by plain torch ─────────────────────────────
def _f64_layer_norm(x, g, b):
    return F.layer_norm(x, (x.shape[-1],), g, b, 1e-5)


def _f64_attention(q, k, v, causal):
    """softmax(q k^T / sqrt(D)) v, query i of the last rows seeing keys j <= i."""
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    if causal:
        Tq, Tk = s.shape[-2:]
        keep = torch.ones(Tq, Tk, dtype=torch.bool, device=s.device).tril(Tk - Tq)
        s = s.masked_fill(~keep, float("-inf"))
    return torch.matmul(torch.softmax(s, -1), v)


def _f64_gpt2(c, i):
    """(logits, keys, values of each layer) of the whole GPT-2."""
    cfg = _config(c)
    dt = getattr(torch, c.get("dtype", "float32"))
    w = {k: t.to(dt).double() for k, t in i["weights"].items()}
    H, d = cfg["n_head"], cfg["n_embd"]
    ids = i["ids"].long()
    decode = c["kind"] == "gpt2_decode"
    ids = ids[:, None] if decode else ids
    B, T = ids.shape
    at = torch.full((1,), c["context"], device="cuda") if decode else torch.arange(T, device="cuda")
    x = w["transformer.wte.weight"][ids] + w["transformer.wpe.weight"][at]
    keys, values = [], []
    for n in range(cfg["n_layer"]):
        p = f"transformer.h.{n}."
        h = _f64_layer_norm(x, w[p + "ln_1.weight"], w[p + "ln_1.bias"])
        qkv = h @ w[p + "attn.c_attn.weight"] + w[p + "attn.c_attn.bias"]
        q, k, v = (t.reshape(B, T, H, d // H).transpose(1, 2).contiguous() for t in qkv.split(d, -1))
        keys.append(k[:, :, 0] if decode else k)
        values.append(v[:, :, 0] if decode else v)
        if decode:
            k, v = torch.cat([i["k"][n].double(), k], 2), torch.cat([i["v"][n].double(), v], 2)
        a = _f64_attention(q, k, v, True).transpose(1, 2).reshape(B, T, d)
        x = x + a @ w[p + "attn.c_proj.weight"] + w[p + "attn.c_proj.bias"]
        h = _f64_layer_norm(x, w[p + "ln_2.weight"], w[p + "ln_2.bias"])
        f = F.gelu(h @ w[p + "mlp.c_fc.weight"] + w[p + "mlp.c_fc.bias"], approximate="tanh")
        x = x + f @ w[p + "mlp.c_proj.weight"] + w[p + "mlp.c_proj.bias"]
    x = _f64_layer_norm(x, w["transformer.ln_f.weight"], w["transformer.ln_f.bias"])
    return (x @ w["transformer.wte.weight"].t()).reshape(B * T, VOCAB), keys, values


def exact(case, seed):
    c, kind = case, case["kind"]
    i = _inputs(c, seed)
    if kind == "mlp_step":
        params = [t.double().requires_grad_(True) for p in i["params"] for t in p]
        h = i["x"].double()
        for n in range(0, len(params), 2):
            h = F.linear(h, params[n], params[n + 1])
            h = torch.relu(h) if n + 2 < len(params) else h
        loss = F.mse_loss(h, i["y"].double())
        grads = torch.autograd.grad(loss, params)
        return [loss.detach().reshape(1)] + [(p - LR * g).detach() for p, g in zip(params, grads)]
    if kind in ("gpt2_forward", "gpt2_prefill", "gpt2_decode"):
        with torch.no_grad():
            logits, keys, values = _f64_gpt2(c, i)
        return [logits] if kind == "gpt2_forward" else [logits] + keys + values
    if kind in ("block_train", "attention_train"):
        s = {k: t.double().requires_grad_(k != "go") for k, t in i.items()}
        if kind == "block_train":
            B, T, d = c["B"], c["T"], c["d"]
            x = s["x"].reshape(B * T, d)
            qkv = F.linear(_f64_layer_norm(x, s["g1"], s["b1"]), s["wqkv"], s["bqkv"]).view(B, T, 3, d // 64, 64)
            q, k, v = (qkv[:, :, j].transpose(1, 2).contiguous() for j in range(3))
            a = _f64_attention(q, k, v, True).transpose(1, 2).reshape(B * T, d)
            x = x + F.linear(a, s["wo"], s["bo"])
            f = F.gelu(F.linear(_f64_layer_norm(x, s["g2"], s["b2"]), s["wfc"], s["bfc"]), approximate="tanh")
            out, wanted = (x + F.linear(f, s["wproj"], s["bproj"])).view(B, T, d), ("x",) + BLOCK
        else:
            out, wanted = _f64_attention(s["q"], s["k"], s["v"], c["causal"]), ("q", "k", "v")
        return [out.detach()] + list(torch.autograd.grad(out, [s[k] for k in wanted], s["go"]))
    if kind == "attention":
        return [_f64_attention(i["q"].double(), i["k"].double(), i["v"].double(), c["causal"])]
    if kind == "linear":
        y = F.linear(i["x"].double(), i["w"].double(), i["b"].double())
        y = torch.relu(y) if c["act"] == "relu" else F.gelu(y, approximate="tanh") if c["act"] == "gelu" else y
        return [y]
    if kind in ("linear_int8", "quantize"):
        w = i["w"]
        scale = w.abs().amax(1) / 127.0   # the codes are defined by the fp32 scale
        codes = torch.clamp(torch.round(w / scale[:, None]), -128, 127)
        deq = codes.double() * scale.double()[:, None]
        if kind == "quantize":
            return [None, scale.double(), deq]
        return [i["x"].double() @ deq.t()]
    if kind == "rows":
        x = i["x"].double()
        if c["op"] == "layer_norm":
            return [_f64_layer_norm(x, i["g"].double(), i["b"].double())]
        return [torch.softmax(x, -1) if c["op"] == "softmax" else torch.log_softmax(x, -1)]
    ids = i["ids"].long()
    grad = torch.zeros(c["vocab"], c["d"], dtype=torch.float64, device="cuda")
    return [i["w"].double()[ids], grad.index_add_(0, ids, i["go"].double())]
