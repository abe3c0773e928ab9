"""The work that users of this framework have it do, as timed cases.

A case is a dict of plain values; its ``kind`` names one of the classes below,
each of which stands for one public entry point with the options used in
earnest: tensor products (``Tensor @``), ``nn.Linear``, ``lm.SwiGLU``, the
attention products, ``lm`` causal grouped-query attention, ``nn`` multi-head
attention in training and with a KV cache, ``lm.SparseMoE`` and a whole
``lm.Decoder.loss`` step.  Sizes are those of this repository's ``Config``
defaults (width 1024, 16 heads of 64 with 4 kv heads, SwiGLU 3584, 8 experts of
1792, vocabulary 32768, sequences up to 1024), of ``bench.py`` and of the tests;
odd ones are mixed in by ``draw``.

``prepare`` draws the inputs on the GPU from the seed and hands them to the
framework as its own storages; ``run`` is one pass through the entry point;
``exact`` computes the same outputs from the same inputs in float64 with plain
torch.
"""
from __future__ import annotations

from math import exp, log, prod, sqrt

import torch
import torch.nn.functional as F

from qutai_amd import Tensor
from qutai_amd.backends import amd, amd_lm
from qutai_amd.lm import Config, Decoder, SparseMoE, SwiGLU, attention_products, autocast
from qutai_amd.lm.layers import attention
from qutai_amd.nn import KVCache, Linear, MultiHeadAttention

TORCH = {"float32": torch.float32, "bfloat16": torch.bfloat16}
RAW = {"float32": ("<f4", torch.float32), "bfloat16": ("<i2", torch.bfloat16)}
BYTES = {"float32": 4, "bfloat16": 2}


# ---- between torch and the framework's storages -----------------------------------

class _Memory:
    """A storage's device memory under the array interface that torch reads."""

    def __init__(self, storage):
        self.storage = storage  # the view keeps the memory alive
        self.__cuda_array_interface__ = {"shape": (storage.size,), "typestr": RAW[storage.dtype][0],
                                         "data": (storage.ptr, False), "strides": None, "version": 2}


def view(storage, shape):
    """The storage's memory as a torch tensor (no copy)."""
    return torch.as_tensor(_Memory(storage), device="cuda").view(RAW[storage.dtype][1]).reshape(shape)


def store(values):
    """A framework storage holding a torch tensor's values."""
    storage = amd.AMDStorage(values.numel(), {t: n for n, t in TORCH.items()}[values.dtype])
    view(storage, values.shape).copy_(values)
    return storage


def tensor(values, grad=False):
    return Tensor(store(values), shape=tuple(values.shape), requires_grad=grad)


class Outputs(dict):
    """Named result Tensors, seen as torch tensors (no copy) when they are
    read: a program of this framework's users keeps them as Tensors, so a pass
    does not pay for the conversion."""

    def __getitem__(self, name):
        value = super().__getitem__(name)
        return view(value.storage, value.shape)


class Draws:
    """Random values on the GPU, from the seed alone."""

    def __init__(self, seed):
        self.generator = torch.Generator(device="cuda")
        self.generator.manual_seed(seed)

    def normal(self, shape, dtype="float32", std=1.0):
        return (torch.randn(shape, generator=self.generator, device="cuda") * std).to(TORCH[dtype])

    def uniform(self, shape, dtype, bound):
        return ((torch.rand(shape, generator=self.generator, device="cuda") * 2 - 1) * bound).to(TORCH[dtype])

    def integers(self, shape, high):
        return torch.randint(high, shape, generator=self.generator, device="cuda")


def wide(inputs, *names):
    """float64 leaves of the named inputs, for the exact gradients."""
    return {n: inputs[n].double().requires_grad_() for n in names}


def linear_of(weight, bias):
    """An nn.Linear that holds the given weights (as after loading them)."""
    layer = Linear(1, 1)
    layer.weight, layer.bias = tensor(weight, True), tensor(bias, True)
    return layer


def log_between(rng, low, high):
    """An integer spread evenly over the logarithm; not only round ones."""
    return max(low, min(high, round(exp(rng.uniform(log(low), log(high))))))


def clear(tensors):
    for t in tensors:
        t.grad = None


# ---- tensor products ------------------------------------------------------------

class Matmul:
    """``a @ b`` of two matrices in one storage type."""

    def inputs(self, c, seed):
        d = Draws(seed)
        return {"a": d.normal((c["m"], c["k"]), c["dtype"], c["k"] ** -0.5), "b": d.normal((c["k"], c["n"]), c["dtype"])}

    def prepare(self, c, x):
        return tensor(x["a"]), tensor(x["b"])

    def run(self, state):
        a, b = state
        return Outputs(out=a @ b)

    def exact(self, c, x):
        return {"out": x["a"].double() @ x["b"].double()}

    def work(self, c):
        m, k, n = c["m"], c["k"], c["n"]
        return (m * k + k * n + m * n) * BYTES[c["dtype"]], 2 * m * k * n

    def draw(self, rng):
        c = {"m": log_between(rng, 32, 4096), "k": log_between(rng, 64, 4096), "n": log_between(rng, 32, 4096)}
        if rng.random() < 0.5:  # widths of real layers
            c["k"], c["n"] = (max(64, v // 64 * 64) for v in (c["k"], c["n"]))
        return {**c, "dtype": rng.choice(["float32", "bfloat16"])}


# ---- layers ---------------------------------------------------------------------

class LinearLayer:
    """``nn.Linear`` with its bias, forward or forward and backward."""

    def inputs(self, c, seed):
        d, t = Draws(seed), c["dtype"]
        i, o = c["inputs"], c["outputs"]
        x = {"x": d.normal((c["rows"], i), t), "weight": d.uniform((i, o), t, i ** -0.5),
             "bias": d.uniform((o,), t, i ** -0.5)}
        if c["train"]:
            x["g"] = d.normal((c["rows"], o), t)
        return x

    def prepare(self, c, x):
        return (linear_of(x["weight"], x["bias"]), tensor(x["x"], c["train"]),
                tensor(x["g"]) if c["train"] else None)

    def run(self, state):
        layer, x, g = state
        clear((x, *layer.parameters()))
        y = layer(x)
        if g is None:
            return Outputs(y=y)
        y.backward(g)
        return Outputs(y=y, dx=x.grad, dw=layer.weight.grad, db=layer.bias.grad)

    def exact(self, c, x):
        v = wide(x, "x", "weight", "bias")
        y = v["x"] @ v["weight"] + v["bias"]
        if not c["train"]:
            return {"y": y.detach()}
        y.backward(x["g"].double())
        return {"y": y.detach(), "dx": v["x"].grad, "dw": v["weight"].grad, "db": v["bias"].grad}

    def work(self, c):
        r, i, o, e = c["rows"], c["inputs"], c["outputs"], BYTES[c["dtype"]]
        forward = (r * i + i * o + o + r * o) * e
        if not c["train"]:
            return forward, 2 * r * i * o
        return forward + (r * o + r * i + i * o + o) * e, 6 * r * i * o

    def draw(self, rng):
        c = {"rows": log_between(rng, 1, 4096), "inputs": log_between(rng, 64, 2048),
             "outputs": log_between(rng, 10, 4096)}
        if rng.random() < 0.5:
            c["inputs"], c["outputs"] = (max(64, c[n] // 64 * 64) for n in ("inputs", "outputs"))
        return {**c, "dtype": rng.choice(["float32", "float32", "bfloat16"]), "train": rng.random() < 0.6}


class _DeviceInit:
    """Builds lm layers without their host-side random draws (every weight is
    replaced afterwards), as a program does that loads its weights."""

    def __enter__(self):
        self.normal = amd_lm.normal
        amd_lm.normal = lambda size, mean=0.0, std=1.0, *, seed=None, dtype="float32": amd.AMDStorage(size, dtype)

    def __exit__(self, *error):
        amd_lm.normal = self.normal


def fill(parameter, values):
    view(parameter.storage, parameter.shape).copy_(values.reshape(parameter.shape))


class SwiGLULayer:
    """``lm.SwiGLU`` forward and backward: fp32 weights and inputs under
    autocast (bf16 products), or fp32 throughout."""

    def inputs(self, c, seed):
        d, w, h = Draws(seed), c["width"], c["hidden"]
        return {"x": d.normal((c["rows"], w)), "gate": d.normal((h, w), std=0.02), "up": d.normal((h, w), std=0.02),
                "down": d.normal((w, h), std=0.02),
                "g": d.normal((c["rows"], w), "bfloat16" if c["autocast"] else "float32")}

    def prepare(self, c, x):
        with _DeviceInit():
            layer = SwiGLU(c["width"], c["hidden"])
        for name in ("gate", "up", "down"):
            fill(getattr(layer, name).weight, x[name])
        return c["autocast"], layer, tensor(x["x"], True), tensor(x["g"])

    def run(self, state):
        cast, layer, x, g = state
        clear((x, *layer.parameters()))
        if cast:
            with autocast():
                y = layer(x)
        else:
            y = layer(x)
        y.backward(g)
        return Outputs(y=y, dx=x.grad, gate=layer.gate.weight.grad, up=layer.up.weight.grad,
                       down=layer.down.weight.grad)

    def exact(self, c, x):
        v = wide(x, "x", "gate", "up", "down")
        y = (F.silu(v["x"] @ v["gate"].T) * (v["x"] @ v["up"].T)) @ v["down"].T
        y.backward(x["g"].double())
        return {"y": y.detach(), "dx": v["x"].grad, **{n: v[n].grad for n in ("gate", "up", "down")}}

    def work(self, c):
        r, w, h = c["rows"], c["width"], c["hidden"]
        e = 2 if c["autocast"] else 4
        return 4 * 2 * r * w + 2 * e * r * w + 4 * 6 * w * h, 18 * r * w * h

    def draw(self, rng):
        cast = rng.random() < 0.7
        return {"rows": log_between(rng, 16, 4096 if cast else 1024), "width": rng.choice([256, 384, 512, 768, 1024]),
                "hidden": rng.choice([512, 1000, 1408, 2048, 3584]), "autocast": cast}


class MoE:
    """``lm.SparseMoE`` forward and backward: bf16 activations over fp32
    weights, or fp32 throughout."""

    def inputs(self, c, seed):
        d, w, h, e = Draws(seed), c["width"], c["hidden"], c["experts"]
        return {"x": d.normal((c["rows"], w), c["dtype"]), "router": d.normal((e, w), std=0.02),
                "gate": d.normal((e, h, w), std=0.02), "up": d.normal((e, h, w), std=0.02),
                "down": d.normal((e, w, h), std=0.02), "g": d.normal((c["rows"], w), c["dtype"])}

    def prepare(self, c, x):
        with _DeviceInit():
            layer = SparseMoE(c["width"], c["hidden"], c["experts"], c["top_k"])
        for parameter, name in zip(layer.parameters(), ("router", "gate", "up", "down")):
            fill(parameter, x[name])
        return layer, tensor(x["x"], True), tensor(x["g"])

    def run(self, state):
        layer, x, g = state
        clear((x, *layer.parameters()))
        y, aux = layer(x)
        y.backward(g)
        grads = dict(zip(("router", "gate", "up", "down"), (p.grad for p in layer.parameters())))
        return Outputs(y=y, aux=aux, dx=x.grad, **grads)

    def exact(self, c, x):
        v = wide(x, "x", "router", "gate", "up", "down")
        probs = (v["x"] @ v["router"].T).softmax(-1)
        top, chosen = probs.topk(c["top_k"], dim=-1)
        weights = top / top.sum(-1, keepdim=True)
        y = torch.zeros_like(v["x"])
        for e in range(c["experts"]):
            row, slot = (chosen == e).nonzero(as_tuple=True)
            part = v["x"][row]
            out = (F.silu(part @ v["gate"][e].T) * (part @ v["up"][e].T)) @ v["down"][e].T
            y = y.index_add(0, row, weights[row, slot, None] * out)
        share = torch.bincount(chosen.reshape(-1), minlength=c["experts"]) / chosen.numel()
        aux = c["experts"] * (share * probs.mean(0)).sum()
        y.backward(x["g"].double())
        return {"y": y.detach(), "aux": aux.detach(), "dx": v["x"].grad,
                **{n: v[n].grad for n in ("router", "gate", "up", "down")}}

    def work(self, c):
        r, w, h, e = c["rows"], c["width"], c["hidden"], c["experts"]
        return 4 * r * w * BYTES[c["dtype"]] + 4 * 2 * e * (3 * h + 1) * w, 18 * r * c["top_k"] * w * h

    def draw(self, rng):
        dtype = rng.choice(["bfloat16", "bfloat16", "float32"])
        return {"rows": log_between(rng, 32, 4096 if dtype == "bfloat16" else 1024),
                "width": rng.choice([256, 512, 1024]), "hidden": rng.choice([256, 704, 1408, 1792]),
                "experts": rng.choice([4, 8, 16]), "top_k": 2, "dtype": dtype}


# ---- attention --------------------------------------------------------------------

def attend(q, k, v, causal):
    """softmax(Q K^T / sqrt(D)) V on (batch, heads, time, dim) float64."""
    scores = (q @ k.transpose(-1, -2)) / sqrt(q.shape[-1])
    if causal:
        time, total = scores.shape[-2:]
        hidden = torch.ones(time, total, dtype=torch.bool, device=q.device).triu(1 + total - time)
        scores = scores.masked_fill(hidden, float("-inf"))
    return scores.softmax(-1) @ v


class Products:
    """``attention_products``: batched scores, row softmax, batched values."""

    def inputs(self, c, seed):
        d, shape = Draws(seed), (c["groups"], c["time"], c["dim"])
        return {n: d.normal(shape, c["dtype"]) for n in "qkv"}

    def prepare(self, c, x):
        return tuple(tensor(x[n]) for n in "qkv")

    def run(self, state):
        out, probs = attention_products(*state)
        return Outputs(out=out, probs=probs)

    def exact(self, c, x):
        q, k, v = (x[n].double() for n in "qkv")
        probs = ((q @ k.transpose(1, 2)) / sqrt(c["dim"])).softmax(-1)
        return {"out": probs @ v, "probs": probs}

    def work(self, c):
        g, t, d, e = c["groups"], c["time"], c["dim"], BYTES[c["dtype"]]
        return (4 * g * t * d + 4 * g * t * t) * e, 4 * g * t * t * d  # scores and probabilities are both stored

    def draw(self, rng):
        time = log_between(rng, 64, 2048)
        most = min(128, 100_000_000 // (time * time))
        return {"groups": log_between(rng, 4, most) if most > 4 else 4, "time": time,
                "dim": rng.choice([32, 64, 64, 128]), "dtype": rng.choice(["float32", "bfloat16", "bfloat16"])}


class GroupedQuery:
    """``lm`` causal grouped-query attention, forward and backward."""

    def inputs(self, c, seed):
        d, rows = Draws(seed), (c["batch"], c["time"])
        q, kv = (*rows, c["heads"] * c["dim"]), (*rows, c["kv_heads"] * c["dim"])
        return {n: d.normal(s, c["dtype"]) for n, s in (("q", q), ("k", kv), ("v", kv), ("g", q))}

    def prepare(self, c, x):
        return c["heads"], c["kv_heads"], *(tensor(x[n], True) for n in "qkv"), tensor(x["g"])

    def run(self, state):
        heads, kv_heads, q, k, v, g = state
        clear((q, k, v))
        out = attention(q, k, v, heads, kv_heads)
        out.backward(g)
        return Outputs(out=out, dq=q.grad, dk=k.grad, dv=v.grad)

    def exact(self, c, x):
        v = wide(x, "q", "k", "v")
        group = c["heads"] // c["kv_heads"]

        def split(t, heads):
            return t.reshape(c["batch"], c["time"], heads, c["dim"]).transpose(1, 2)

        k, val = (split(v[n], c["kv_heads"]).repeat_interleave(group, dim=1) for n in "kv")
        out = attend(split(v["q"], c["heads"]), k, val, True).transpose(1, 2).reshape(x["q"].shape)
        out.backward(x["g"].double())
        return {"out": out.detach(), "dq": v["q"].grad, "dk": v["k"].grad, "dv": v["v"].grad}

    def work(self, c):
        rows, pairs = c["batch"] * c["time"], c["batch"] * c["heads"] * c["time"] * (c["time"] + 1) // 2
        values = rows * c["dim"] * (4 * c["heads"] + 4 * c["kv_heads"])
        return values * BYTES[c["dtype"]], 14 * pairs * c["dim"]

    def draw(self, rng):
        time = log_between(rng, 40, 1024)
        heads = rng.choice([4, 8, 12, 16])
        return {"batch": rng.randint(1, 4), "time": time, "heads": heads, "kv_heads": heads // rng.choice([1, 2, 4]),
                "dim": rng.choice([32, 64, 64, 80, 96, 128, 128]),
                "dtype": rng.choice(["bfloat16", "bfloat16", "float32"])}


class MultiHead:
    """``nn.MultiHeadAttention``: a training pass over whole sequences, or
    (``past`` > 0) inference of new positions with a KV cache."""

    NAMES = ("query", "key", "value", "output")
    # what a training pass leaves beside y and dx; not the key bias, which
    # shifts every score of a row alike: its gradient is rounding and no more
    GRADS = tuple((n, p) for n in NAMES for p in ("weight", "bias") if (n, p) != ("key", "bias"))

    def inputs(self, c, seed):
        d, f, t = Draws(seed), c["features"], c["dtype"]
        shape = (c["batch"], c["time"], f)
        x = {"x": d.normal(shape, t)}
        for name in self.NAMES:
            x[name] = d.uniform((f, f), t, f ** -0.5)
            x[name + "_bias"] = d.uniform((f,), t, f ** -0.5)
        if c["past"]:
            for name in ("keys", "values"):
                x[name] = d.normal((c["batch"], c["heads"], c["past"], f // c["heads"]), t)
        else:
            x["g"] = d.normal(shape, t)
        return x

    def prepare(self, c, x):
        layer = MultiHeadAttention(c["heads"], c["heads"], causal=c["causal"])
        for name in self.NAMES:
            setattr(layer, name, linear_of(x[name], x[name + "_bias"]))
        if c["past"]:
            return layer, tensor(x["x"]), tensor(x["keys"]), tensor(x["values"]), None
        return layer, tensor(x["x"], True), None, None, tensor(x["g"])

    def run(self, state):
        layer, x, keys, values, g = state
        if g is None:
            cache = KVCache()
            cache.keys, cache.values = keys, values
            return Outputs(y=layer(x, cache=cache), keys=cache.keys, values=cache.values)
        clear((x, *layer.parameters()))
        y = layer(x)
        y.backward(g)
        grads = {f"{n}_{p}": getattr(getattr(layer, n), p).grad for n, p in self.GRADS}
        return Outputs(y=y, dx=x.grad, **grads)

    def exact(self, c, x):
        v = wide(x, "x", *self.NAMES, *(n + "_bias" for n in self.NAMES))
        batch, time, f = x["x"].shape

        def project(name, values):
            return values @ v[name] + v[name + "_bias"]

        q, k, val = (project(n, v["x"]).reshape(batch, time, c["heads"], -1).transpose(1, 2)
                     for n in ("query", "key", "value"))
        if c["past"]:
            k, val = (torch.cat((x[n].double(), new), 2) for n, new in (("keys", k), ("values", val)))
        y = project("output", attend(q, k, val, c["causal"]).transpose(1, 2).reshape(batch, time, f))
        if c["past"]:
            return {"y": y.detach(), "keys": k.detach(), "values": val.detach()}
        y.backward(x["g"].double())
        grads = {f"{n}_{p}": v[n if p == "weight" else n + "_bias"].grad for n, p in self.GRADS}
        return {"y": y.detach(), "dx": v["x"].grad, **grads}

    def work(self, c):
        rows, f, e = c["batch"] * c["time"], c["features"], BYTES[c["dtype"]]
        if c["past"]:
            cache = 2 * c["batch"] * (2 * c["past"] + c["time"]) * f  # read, and written with the new positions
            pairs = rows * (c["past"] + c["time"])
            return (2 * rows * f + 4 * (f + 1) * f + cache) * e, 8 * rows * f * f + 4 * pairs * f
        pairs = c["batch"] * (c["time"] * (c["time"] + 1) // 2 if c["causal"] else c["time"] ** 2)
        return (4 * rows * f + 8 * (f + 1) * f) * e, 24 * rows * f * f + 14 * pairs * f

    def draw(self, rng):
        dim = rng.choice([32, 64, 64, 128])
        heads = rng.choice([4, 8, 16]) if dim < 128 else rng.choice([2, 4, 8])
        c = {"batch": rng.randint(1, 16), "features": dim * heads, "heads": heads}
        if rng.random() < 0.5:
            return {**c, "time": rng.choice([1, 1, 1, 4, 7]), "past": log_between(rng, 15, 2048), "causal": True,
                    "dtype": rng.choice(["bfloat16", "bfloat16", "float32"])}
        return {**c, "batch": min(8, c["batch"]), "time": log_between(rng, 17, 512), "past": 0,
                "causal": rng.random() < 0.5, "dtype": rng.choice(["float32", "float32", "bfloat16"])}


# ---- a whole model -----------------------------------------------------------------

class DecoderLoss:
    """``lm.Decoder.loss`` under autocast, forward and backward: embedding,
    norms, rotary attention, SwiGLU, the chunked head and every gradient."""

    def config(self, c):
        return Config(vocab_size=c["vocab"], n_layers=c["layers"], d_model=c["width"], n_heads=c["heads"],
                      n_kv_heads=c["kv_heads"], d_ff=c["hidden"], max_seq_len=c["time"])

    def inputs(self, c, seed):
        d, w, h = Draws(seed), c["width"], c["hidden"]
        kv, small = c["kv_heads"] * (w // c["heads"]), 0.02 / sqrt(2 * c["layers"])
        x = {"tokens": d.integers((c["batch"], c["time"]), c["vocab"]),
             "embedding.weight": d.normal((c["vocab"], w), std=0.02)}
        for i in range(c["layers"]):
            p = f"blocks.{i}."
            x[p + "attn_norm.weight"] = 1 + d.normal((w,), std=0.05)
            x[p + "ffn_norm.weight"] = 1 + d.normal((w,), std=0.05)
            for name, rows, std in (("q", w, 0.02), ("k", kv, 0.02), ("v", kv, 0.02), ("out", w, small)):
                x[p + f"attn.{name}.weight"] = d.normal((rows, w), std=std)
            for name, shape, std in (("gate", (h, w), 0.02), ("up", (h, w), 0.02), ("down", (w, h), small)):
                x[p + f"ffn.{name}.weight"] = d.normal(shape, std=std)
        x["norm.weight"] = 1 + d.normal((w,), std=0.05)
        return x

    def prepare(self, c, x):
        with _DeviceInit():
            model = Decoder(self.config(c))
        for name, parameter in model.named_parameters():
            fill(parameter, x[name])
        return model, x["tokens"].tolist()

    def run(self, state):
        model, tokens = state
        clear(model.parameters())
        with autocast():
            loss = model.loss(tokens)
        loss.backward()
        return Outputs(loss=loss, **{n: p.grad for n, p in model.named_parameters()})

    def exact(self, c, x):
        v = wide(x, *(n for n in x if n != "tokens"))
        batch, time, w = c["batch"], c["time"], c["width"]
        dim, group = w // c["heads"], c["heads"] // c["kv_heads"]
        config = self.config(c)
        pairs = torch.arange(0, dim, 2, device="cuda", dtype=torch.float64)
        angle = torch.arange(time, device="cuda", dtype=torch.float64)[:, None] * config.rope_theta ** (-pairs / dim)
        cos, sin = angle.cos(), angle.sin()

        def norm(values, weight):
            return values * (values.square().mean(-1, keepdim=True) + config.norm_eps).rsqrt() * weight

        def heads(values, count):
            return values.reshape(batch, time, count, dim).transpose(1, 2)

        def rotate(values):
            even, odd = values[..., 0::2], values[..., 1::2]
            return torch.stack((even * cos - odd * sin, even * sin + odd * cos), -1).flatten(-2)

        hidden = v["embedding.weight"][x["tokens"]]
        for i in range(c["layers"]):
            p = f"blocks.{i}."
            y = norm(hidden, v[p + "attn_norm.weight"])
            q = rotate(heads(y @ v[p + "attn.q.weight"].T, c["heads"]))
            k = rotate(heads(y @ v[p + "attn.k.weight"].T, c["kv_heads"])).repeat_interleave(group, 1)
            val = heads(y @ v[p + "attn.v.weight"].T, c["kv_heads"]).repeat_interleave(group, 1)
            mixed = attend(q, k, val, True).transpose(1, 2).reshape(batch, time, w)
            hidden = hidden + mixed @ v[p + "attn.out.weight"].T
            y = norm(hidden, v[p + "ffn_norm.weight"])
            act = F.silu(y @ v[p + "ffn.gate.weight"].T) * (y @ v[p + "ffn.up.weight"].T)
            hidden = hidden + act @ v[p + "ffn.down.weight"].T
        logits = norm(hidden, v["norm.weight"])[:, :-1] @ v["embedding.weight"].T
        loss = F.cross_entropy(logits.reshape(-1, c["vocab"]), x["tokens"][:, 1:].reshape(-1))
        loss.backward()
        return {"loss": loss.detach(), **{n: t.grad for n, t in v.items()}}

    def _weights(self, c):
        w = c["width"]
        return c["layers"] * (2 * w * w + 2 * w * c["kv_heads"] * (w // c["heads"]) + 3 * w * c["hidden"])

    def work(self, c):
        tokens, weights = c["batch"] * c["time"], self._weights(c) + c["vocab"] * c["width"]
        pairs = c["layers"] * c["batch"] * c["time"] * (c["time"] + 1) // 2
        return 4 * 2 * weights, 6 * weights * tokens + 14 * pairs * c["width"]

    def draw(self, rng):
        dim, heads = rng.choice([64, 64, 128]), rng.choice([4, 8])
        return {"layers": rng.randint(1, 2), "batch": rng.randint(1, 4), "time": log_between(rng, 33, 512),
                "width": dim * heads, "heads": heads, "kv_heads": heads // rng.choice([1, 2, 4]),
                "hidden": rng.choice([704, 1408, 2048]), "vocab": rng.choice([1000, 8192, 32768])}


KINDS = {"matmul": Matmul(), "linear": LinearLayer(), "swiglu": SwiGLULayer(), "moe": MoE(), "products": Products(),
         "grouped_query": GroupedQuery(), "multi_head": MultiHead(), "decoder_loss": DecoderLoss()}


def listed():
    return [
        # the smallest call: one layer of a small network, where latency counts
        {"name": "linear_small_fp32", "kind": "linear", "rows": 128, "inputs": 256, "outputs": 64, "dtype": "float32",
         "train": False},
        # training a feed-forward layer in the default storage type
        {"name": "linear_train_fp32", "kind": "linear", "rows": 2048, "inputs": 1024, "outputs": 3584,
         "dtype": "float32", "train": True},
        # the headline product, and an odd-sized one in the default storage type
        {"name": "matmul_bf16_square", "kind": "matmul", "m": 4096, "k": 4096, "n": 4096, "dtype": "bfloat16"},
        {"name": "matmul_fp32_ragged", "kind": "matmul", "m": 4095, "k": 1000, "n": 4097, "dtype": "float32"},
        # a decoder's feed-forward layer in mixed-precision training, Config's widths
        {"name": "swiglu_train_bf16", "kind": "swiglu", "rows": 4096, "width": 1024, "hidden": 3584, "autocast": True},
        # attention whose probabilities are kept, bench.py's shape
        {"name": "attention_products_bf16", "kind": "products", "groups": 128, "time": 2048, "dim": 64,
         "dtype": "bfloat16"},
        # a decoder's attention in mixed-precision training: Config's heads of 64, and heads of 128
        {"name": "attention_train_d64", "kind": "grouped_query", "batch": 8, "time": 1024, "heads": 16, "kv_heads": 4,
         "dim": 64, "dtype": "bfloat16"},
        {"name": "attention_train_d128", "kind": "grouped_query", "batch": 4, "time": 1024, "heads": 16, "kv_heads": 4,
         "dim": 128, "dtype": "bfloat16"},
        # a multi-head layer trained in the default storage type
        {"name": "mha_train_fp32", "kind": "multi_head", "batch": 8, "time": 512, "features": 512, "heads": 8,
         "past": 0, "causal": True, "dtype": "float32"},
        # generating one position for a batch of sequences
        {"name": "mha_decode_bf16", "kind": "multi_head", "batch": 8, "time": 1, "features": 1024, "heads": 16,
         "past": 1000, "causal": True, "dtype": "bfloat16"},
        # a mixture-of-experts layer in mixed-precision training, Config's experts
        {"name": "moe_train_bf16", "kind": "moe", "rows": 4096, "width": 1024, "hidden": 1792, "experts": 8, "top_k": 2,
         "dtype": "bfloat16"},
        # one training step of a small decoder, everything in it
        {"name": "decoder_loss", "kind": "decoder_loss", "layers": 2, "batch": 4, "time": 512, "width": 1024,
         "heads": 16, "kv_heads": 4, "hidden": 3584, "vocab": 32768},
    ]


def draw(rng):
    kind = rng.choice(sorted(KINDS))
    return {"kind": kind, **KINDS[kind].draw(rng)}


def prepare(case, seed):
    kind = KINDS[case["kind"]]
    return kind, kind.prepare(case, kind.inputs(case, seed))


def run(state):
    kind, inner = state
    return kind.run(inner)


def exact(case, seed):
    kind = KINDS[case["kind"]]
    return kind.exact(case, kind.inputs(case, seed))


def work(case):
    moved, flops = KINDS[case["kind"]].work(case)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    if case["kind"] == "decoder_loss":
        return {"rel": 3e-2}  # bf16 roundings of one layer travel through those after it
    low = case.get("dtype") == "bfloat16" or case.get("autocast")
    return {"rel": 1e-2} if low else {"rel": 1e-5}
