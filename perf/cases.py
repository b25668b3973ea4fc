"""The work a user of this framework has it do, as cases that can be timed and compared.

A case goes through dtmi's public entry points only: the DDP training step, GPT
and Block forward and backward, causal_attention, linear, cross_entropy, the
Tensor operators and the optimizer pass over replica gradients. `prepare` makes
what a user's program holds before the call (arrays, modules, optimizer state,
token ids in HBM), `run` is one pass, `exact` the same numbers in float64 from
plain torch. Inputs come from torch generators seeded with the case's seed.

Ranges (`draw`): sequence lengths, row counts and layer widths are any whole
numbers, not only multiples of a tile; head dimensions 32 to 128; vocabularies
from a character set to 50,304; float32 (both GEMM arithmetics) and float64.
"""
from __future__ import annotations

import contextlib
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parents[1] / "distributed-training_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

from dtmi import _lib, autograd as A, device as dev, nn as N, optim as O, train as S  # noqa: E402
from dtmi.ddp import DDP  # noqa: E402
from dtmi.replicas import SimGroup, ring_segments  # noqa: E402


# ------------------------------------------------------------------- cases
def listed():
    return [
        # dtrain's default training configuration (its driver's flags: dim 128,
        # 4 layers, 4 heads, ctx 64, batch 8, a character vocabulary), two
        # data-parallel replicas: many short launches, loss and norm logged
        # every step as the driver does
        dict(name="train_char", kind="train", dtype="float32", world=2, batch=8, ctx=64, dim=128, heads=4, layers=4,
             vocab=65),
        # validation logits of a small character model on one odd-length text:
        # the smallest call, forward only
        dict(name="logits_one_text", kind="logits", dtype="float32", batch=1, ctx=201, dim=384, heads=6, layers=6,
             vocab=65),
        # one GPT-2-small-shape block on a replica's batch, the layer that the
        # benchmark's step repeats
        dict(name="block_8x1024", kind="block", dtype="float32", math="f32", batch=8, ctx=1024, dim=768, heads=12),
        # the same layer on text that was not cut to a multiple of the tile
        dict(name="block_ragged", kind="block", dtype="float32", math="f32", batch=5, ctx=499, dim=768, heads=12),
        # float64, the type of the parity and checkpoint runs
        dict(name="block_float64", kind="block", dtype="float64", math="f32", batch=4, ctx=250, dim=256, heads=8),
        # short-sequence attention, forward and backward (the attention
        # microbenchmark's shape)
        dict(name="attention_short", kind="attention", dtype="float32", batch=16, heads=12, ctx=256, hdim=64),
        # long sequences with wide heads
        dict(name="attention_wide", kind="attention", dtype="float32", batch=2, heads=8, ctx=2000, hdim=128),
        # a Linear with the split-bf16 arithmetic, the LayerNorm + Linear
        # microbenchmark's shape
        dict(name="linear_bf16x6", kind="linear", dtype="float32", math="bf16x6", rows=16384, nin=768, nout=3072),
        # a Linear of odd sizes, as a user's own model has them
        dict(name="linear_odd", kind="linear", dtype="float32", math="f32", rows=1001, nin=515, nout=1030),
        # the vocabulary head with its loss: 50,257 is GPT-2's vocabulary
        # before padding
        dict(name="head_50257", kind="head", dtype="float32", rows=4096, dim=768, vocab=50257),
        # fixed-order average of 4 replicas, global norm, clip, AdamW over
        # GPT-2-small's parameter count (the bucket + AdamW microbenchmark)
        dict(name="update_124m", kind="update", dtype="float32", world=4, n=124_439_808),
        # a user's own model and loss written with the Tensor operators
        dict(name="operators", kind="operators", dtype="float32", rows=600, nin=100, hidden=300, nout=20),
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["train", "logits", "block", "block", "attention", "attention", "linear", "linear", "head",
                       "update", "operators"])
    f64 = rng.random() < 0.2
    dtype = "float64" if f64 else "float32"
    if kind == "train":
        hd = rng.choice([32, 64])
        heads = rng.randint(1, 6 if hd == 32 else 4)
        return dict(kind=kind, dtype="float32", world=rng.randint(1, 3), batch=rng.randint(2, 12),
                    ctx=_between(rng, 24, 160), dim=hd * heads, heads=heads, layers=rng.randint(2, 4),
                    vocab=_between(rng, 60, 2000))
    if kind == "logits":
        hd = rng.choice([32, 64])
        heads = rng.randint(2, 8)
        return dict(kind=kind, dtype="float32", batch=rng.randint(1, 4), ctx=_between(rng, 16, 512), dim=hd * heads,
                    heads=heads, layers=rng.randint(2, 6), vocab=_between(rng, 60, 5000))
    if kind == "block":
        hd = rng.choice([32, 64, 64, 128])
        heads = rng.randint(2, 8 if hd == 128 or f64 else 12)
        ctx = _between(rng, 32, 512 if f64 else 1024)
        return dict(kind=kind, dtype=dtype, math="f32" if f64 else rng.choice(["f32", "f32", "bf16x6"]),
                    batch=max(1, min(16, _between(rng, 256, 4096 if f64 else 8192) // ctx)), ctx=ctx, dim=hd * heads,
                    heads=heads)
    if kind == "attention":
        hd = rng.choice([32, 64, 64, 80, 96, 128])
        ctx = _between(rng, 32, 700 if f64 else 2048)
        return dict(kind=kind, dtype=dtype, batch=max(1, min(16, _between(rng, 1024, 8192) // ctx)),
                    heads=rng.randint(2, 8 if f64 else 12), ctx=ctx, hdim=hd)
    if kind == "linear":
        return dict(kind=kind, dtype=dtype, math="f32" if f64 else rng.choice(["f32", "f32", "bf16x6"]),
                    rows=_between(rng, 32, 3000 if f64 else 10000), nin=_between(rng, 48, 2048 if f64 else 3072),
                    nout=_between(rng, 48, 2048 if f64 else 3072))
    if kind == "head":
        return dict(kind=kind, dtype="float32", rows=_between(rng, 128, 3000), dim=_between(rng, 64, 768),
                    vocab=_between(rng, 1000, 50304))
    if kind == "update":
        return dict(kind=kind, dtype=dtype, world=rng.randint(2, 4), n=_between(rng, 100_000, 50_000_000))
    return dict(kind=kind, dtype=dtype, rows=_between(rng, 64, 1000), nin=_between(rng, 10, 400),
                hidden=_between(rng, 32, 600), nout=rng.randint(1, 40))


# ------------------------------------------------------------------ inputs
def _torch_dtype(case):
    return torch.float64 if case["dtype"] == "float64" else torch.float32


class _Memory:
    """A DeviceArray's HBM as torch takes it (no copy; keeps the array alive)."""

    def __init__(self, a):
        self.array = a
        self.__cuda_array_interface__ = {"shape": a.shape, "typestr": a.dtype.str, "data": (a.ptr, False),
                                         "strides": None, "version": 2}


def _tensor(a):
    """A contiguous DeviceArray as a torch tensor over the same memory."""
    return torch.as_tensor(_Memory(a), device="cuda")


def _array(t):
    """A DeviceArray with the values of a torch tensor."""
    a = dev.empty(tuple(t.shape), str(t.dtype).split(".")[1])
    _tensor(a).copy_(t)
    return a


def _params(case):
    """(name, shape, mean, deviation) of every parameter, in the modules' order."""
    C = case["dim"]
    L = case.get("layers", 1)

    def block(p):
        return [(p + "ln1.w", (C,), 1, .1), (p + "ln1.b", (C,), 0, .02), (p + "qkv.w", (C, 3 * C), 0, .02),
                (p + "qkv.b", (3 * C,), 0, .02), (p + "proj.w", (C, C), 0, .02 / math.sqrt(2 * L)),
                (p + "proj.b", (C,), 0, .02), (p + "ln2.w", (C,), 1, .1), (p + "ln2.b", (C,), 0, .02),
                (p + "fc.w", (C, 4 * C), 0, .02), (p + "fc.b", (4 * C,), 0, .02),
                (p + "out.w", (4 * C, C), 0, .02 / math.sqrt(2 * L)), (p + "out.b", (C,), 0, .02)]
    if case["kind"] == "block":
        return block("")
    spec = [("tok", (case["vocab"], C), 0, .02), ("pos", (case["ctx"], C), 0, .01)]
    for i in range(L):
        spec += block(f"blocks.{i}.")
    return spec + [("ln.w", (C,), 1, .1), ("ln.b", (C,), 0, .02), ("head.w", (C, case["vocab"]), 0, .02)]


def _inputs(case, seed):
    """The case's inputs as torch tensors on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    dt = _torch_dtype(case)

    def normal(*shape, std=1.0, mean=0.0):
        return torch.randn(shape, generator=g, device="cuda", dtype=dt) * std + mean

    def ids(n, *shape):
        return torch.randint(0, n, shape, generator=g, device="cuda")

    k = case["kind"]
    if k in ("train", "logits", "block"):
        P = {name: normal(*shape, std=sd, mean=m) for name, shape, m, sd in _params(case)}
        if k == "block":
            shape = (case["batch"], case["ctx"], case["dim"])
            return dict(P=P, x=normal(*shape), g=normal(*shape))
        W = case.get("world", 1)
        return dict(P=P, x=ids(case["vocab"], W, case["batch"], case["ctx"]),
                    y=ids(case["vocab"], W, case["batch"], case["ctx"]))
    if k == "attention":
        shape = (case["batch"], case["heads"], case["ctx"], case["hdim"])
        return {n: normal(*shape) for n in "qkvg"}
    if k == "linear":
        return dict(x=normal(case["rows"], case["nin"]), w=normal(case["nin"], case["nout"], std=.02),
                    b=normal(case["nout"], std=.02), g=normal(case["rows"], case["nout"]))
    if k == "head":
        return dict(x=normal(case["rows"], case["dim"]), w=normal(case["dim"], case["vocab"], std=.02),
                    y=ids(case["vocab"], case["rows"]))
    if k == "update":
        n, W = case["n"], case["world"]
        p = normal(n, std=.02)
        rows = torch.empty((W, n), device="cuda", dtype=dt)
        for r in range(W):
            rows[r].normal_(0, 5e-4, generator=g)
        return dict(p=p, rows=rows)
    r, i, h, o = case["rows"], case["nin"], case["hidden"], case["nout"]
    return dict(x=normal(r, i), t=normal(r, o), w1=normal(i, h, std=i ** -.5), b1=normal(h, std=.1),
                w2=normal(h, o, std=h ** -.5), b2=normal(o, std=.1))


# ----------------------------------------------------------- prepare and run
_LR, _BETAS, _EPS, _WD, _CLIP = 1e-3, (0.9, 0.95), 1e-8, 0.1, 1.0


def _config(case):
    return N.GPTConfig(vocab=case.get("vocab", 65), ctx=case["ctx"], dim=case["dim"], heads=case["heads"],
                       layers=case.get("layers", 1), dtype=case["dtype"])


def _load(module, P):
    for name, p in module.named_parameters():
        _tensor(p.data).copy_(P[name])


def prepare(case, seed):
    torch.cuda.synchronize()  # nothing queued still uses memory that torch writes below
    _lib.lib()
    t = _inputs(case, seed)
    k = case["kind"]
    s = {"kind": k, "math": case.get("math", "f32")}
    if k in ("train", "logits"):
        model = N.GPT(_config(case), seed=0)
        _lib.sync()
        _load(model, t["P"])
        s["model"] = model
        x, y = t["x"].cpu().numpy(), t["y"].cpu().numpy()
        if k == "logits":
            s["x"] = A.Indices(x[0])
        else:
            s["ddp"] = DDP(model, SimGroup(case["world"]))
            s["opt"] = O.AdamW([p.data for p in model.parameters()], lr=_LR, betas=_BETAS, eps=_EPS, weight_decay=_WD)
            s["batches"] = [[(A.Indices(x[r]), A.Indices(y[r]))] for r in range(case["world"])]
    elif k == "block":
        s["block"] = N.Block(_config(case), np.random.default_rng(0))
        _lib.sync()
        _load(s["block"], t["P"])
        # every parameter's gradient has its place in one buffer, as DDP lays them out
        ps = s["block"].parameters()
        s["grads"] = dev.empty((sum(p.data.size for p in ps),), case["dtype"])
        off = 0
        for p in ps:
            p.grad_dest = s["grads"][off:off + p.data.size].reshape(p.shape)
            off += p.data.size
        s["x"], s["g"] = _array(t["x"]), _array(t["g"])
    elif k == "head":
        s["x"], s["w"], s["y"] = _array(t["x"]), _array(t["w"]), A.Indices(t["y"].cpu().numpy())
    elif k == "update":
        n = case["n"]
        s["p"], s["rows"] = _array(t["p"]), _array(t["rows"])
        s["pg"], s["segments"] = SimGroup(case["world"]), ring_segments([n], case["world"])
        s["avg"] = dev.empty((n,), case["dtype"])
        s["opt"] = O.AdamW([s["p"]], lr=_LR, betas=_BETAS, eps=_EPS, weight_decay=_WD)
    else:
        s.update({name: _array(v) for name, v in t.items()})
    torch.cuda.synchronize()
    return s


def _leaf(a):
    return A.Tensor(a, requires_grad=True)


def run(s):
    k = s["kind"]
    if k == "train":  # one step of dtmi.train's driver loop
        res = S.step_ddp(s["model"], s["ddp"], s["opt"], s["batches"], clip=_CLIP)
        return {"loss": res.loss, "norm": res.grad_norm, "grads": _tensor(s["ddp"].avg)}
    if k == "logits":
        with A.no_grad():
            return _tensor(s["model"](s["x"]).data)
    math_mode = _lib.use_gemm_math(s["math"]) if s["math"] != "f32" else contextlib.nullcontext()
    if k == "block":
        x = _leaf(s["x"])
        s["block"].zero_grad()
        with math_mode:
            y = s["block"](x)
            y.backward(s["g"])
        return [_tensor(y.data), _tensor(x.grad), _tensor(s["grads"])]
    if k == "attention":
        q, kk, v = _leaf(s["q"]), _leaf(s["k"]), _leaf(s["v"])
        o = A.causal_attention(q, kk, v)
        o.backward(s["g"])
        return [_tensor(a) for a in (o.data, q.grad, kk.grad, v.grad)]
    if k == "linear":
        x, w, b = _leaf(s["x"]), _leaf(s["w"]), _leaf(s["b"])
        with math_mode:
            y = N.linear(x, w, b)
            y.backward(s["g"])
        return [_tensor(a) for a in (y.data, x.grad, w.grad, b.grad)]
    if k == "head":
        x, w = _leaf(s["x"]), _leaf(s["w"])
        z = N.linear(x, w, None)
        loss = A.cross_entropy(z, s["y"])
        loss.backward()
        return [_tensor(a) for a in (z.data, loss.data, x.grad, w.grad)]
    if k == "update":
        s["pg"].average(s["avg"], s["rows"], segments=s["segments"])
        scale, norm = O.clip_scale_device(O.grad_sq_norm([s["avg"]]), _CLIP)
        s["opt"].step([s["avg"]], grad_scale=scale)
        return [_tensor(a) for a in (s["avg"], norm, s["p"], s["opt"].m[0], s["opt"].v[0])]
    w1, b1, w2, b2 = (_leaf(s[n]) for n in ("w1", "b1", "w2", "b2"))
    x, t = A.Tensor(s["x"]), A.Tensor(s["t"])
    err = (x @ w1 + b1).gelu() @ w2 + b2 - t
    loss = (err * err).mean()
    loss.backward()
    return [_tensor(a) for a in (loss.data, w1.grad, b1.grad, w2.grad, b2.grad)]


# ------------------------------------------------------------------- work
def work(case):
    """One pass: inputs read once, outputs written once; products, forward and backward."""
    k = case["kind"]
    es = 8 if case["dtype"] == "float64" else 4
    if k in ("train", "logits", "block"):
        C, T, B = case["dim"], case["ctx"], case["batch"]
        L = case.get("layers", 1)
        M = B * T
        fwd = L * (2 * M * 12 * C * C + 2 * B * T * (T + 1) * C)
        n = L * (12 * C * C + 13 * C)
        if k == "block":
            return {"bytes": es * (2 * n + 4 * M * C), "flops": 3 * fwd}
        V = case["vocab"]
        n += C * (2 * V + T + 2)
        fwd += 2 * M * C * V
        if k == "logits":
            return {"bytes": es * (n + M * V), "flops": fwd}
        W = case["world"]
        return {"bytes": es * n * (W * 2 + 7), "flops": 3 * fwd * W}
    if k == "attention":
        B, H, T, D = (case[x] for x in ("batch", "heads", "ctx", "hdim"))
        return {"bytes": es * 8 * B * H * T * D, "flops": 7 * B * H * T * (T + 1) * D}
    if k == "linear":
        M, K, F = case["rows"], case["nin"], case["nout"]
        return {"bytes": es * (2 * M * K + 2 * K * F + 2 * M * F + 2 * F), "flops": 6 * M * K * F}
    if k == "head":
        M, K, V = case["rows"], case["dim"], case["vocab"]
        return {"bytes": es * (2 * M * K + 2 * K * V + M * V) + 8 * M, "flops": 6 * M * K * V}
    if k == "update":
        return {"bytes": es * case["n"] * (case["world"] + 7), "flops": 20 * case["n"]}
    r, i, h, o = case["rows"], case["nin"], case["hidden"], case["nout"]
    return {"bytes": es * (r * (i + o) + 2 * (i * h + h + h * o + o)), "flops": 2 * r * (2 * i * h + 3 * h * o)}


def tolerance(case):
    """Largest error another correct implementation of the same precision shows."""
    if case["dtype"] == "float64":
        return {"rel": 2e-14}
    # about four times the error against float64 seen over the ranges (the
    # head's input gradient sums over the whole vocabulary)
    return {"train": {"rel": 5e-6}, "logits": {"rel": 5e-6}, "block": {"rel": 5e-6}, "attention": {"rel": 3e-6},
            "linear": {"rel": 4e-6}, "head": {"rel": 8e-6}, "update": {"rel": 1e-6},
            "operators": {"rel": 4e-6}}[case["kind"]]


# ------------------------------------------------------------------ exact
def _ln(x, w, b):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + 1e-5) * w + b


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _attend(q, k, v):
    """Causal attention of one batch element's heads [H, T, D]."""
    T = q.shape[-2]
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    mask = torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1)
    return torch.matmul(torch.softmax(s.masked_fill(mask, float("-inf")), -1), v)


def _block(x, P, p, heads):
    B, T, C = x.shape
    qkv = _ln(x, P[p + "ln1.w"], P[p + "ln1.b"]) @ P[p + "qkv.w"] + P[p + "qkv.b"]
    q, k, v = (t.reshape(B, T, heads, C // heads).permute(0, 2, 1, 3).contiguous() for t in qkv.split(C, dim=-1))
    a = torch.stack([_attend(q[i], k[i], v[i]) for i in range(B)])
    x = x + (a.permute(0, 2, 1, 3).reshape(B, T, C) @ P[p + "proj.w"] + P[p + "proj.b"])
    h = _ln(x, P[p + "ln2.w"], P[p + "ln2.b"]) @ P[p + "fc.w"] + P[p + "fc.b"]
    return x + (_gelu(h) @ P[p + "out.w"] + P[p + "out.b"])


def _gpt(ids, P, case):
    x = P["tok"][ids] + P["pos"][:ids.shape[1]]
    for i in range(case["layers"]):
        x = _block(x, P, f"blocks.{i}.", case["heads"])
    return _ln(x, P["ln.w"], P["ln.b"]) @ P["head.w"]


def exact(case, seed):
    t = _inputs(case, seed)
    k = case["kind"]

    def up(v):
        return v.double() if v.is_floating_point() else v

    if k in ("train", "logits", "block"):
        P = {n: up(v).requires_grad_(k != "logits") for n, v in t.pop("P").items()}
        flat = lambda gs: torch.cat([v.reshape(-1) for v in gs])  # noqa: E731
        if k == "logits":
            return _gpt(t["x"][0], P, case)
        if k == "block":
            x = up(t["x"]).requires_grad_(True)
            y = _block(x, P, "", case["heads"])
            gs = torch.autograd.grad(y, [x] + list(P.values()), up(t["g"]))
            return [y.detach(), gs[0], flat(gs[1:])]
        W, total, loss = case["world"], None, 0.0
        for r in range(W):
            z = _gpt(t["x"][r], P, case).reshape(-1, case["vocab"])
            l = torch.nn.functional.cross_entropy(z, t["y"][r].reshape(-1))
            gr = flat(torch.autograd.grad(l, list(P.values())))
            total = gr if total is None else total + gr
            loss += float(l)
        avg = total / W
        return {"loss": loss / W, "norm": float(avg.norm()), "grads": avg}
    t = {n: up(v) for n, v in t.items()}
    if k == "attention":
        leaves = [t[n].requires_grad_(True) for n in "qkv"]
        o = torch.stack([_attend(*(x[i] for x in leaves)) for i in range(case["batch"])])
        return [o.detach(), *torch.autograd.grad(o, leaves, t["g"])]
    if k == "linear":
        return [t["x"] @ t["w"] + t["b"], t["g"] @ t["w"].T, t["x"].T @ t["g"], t["g"].sum(0)]
    if k == "head":
        x, w = t["x"], t["w"]
        z = x @ w
        loss = torch.nn.functional.cross_entropy(z, t["y"])
        d = torch.softmax(z, -1)
        d[torch.arange(case["rows"], device="cuda"), t["y"]] -= 1
        d /= case["rows"]
        return [z, loss, d @ w.T, x.T @ d]
    if k == "update":
        avg = t["rows"].sum(0) / case["world"]
        norm = avg.norm()
        g = avg * (1.0 if float(norm) <= _CLIP else _CLIP / (float(norm) + 1e-6))
        m, v = (1 - _BETAS[0]) * g, (1 - _BETAS[1]) * g * g
        p = t["p"] - _LR * ((m / (1 - _BETAS[0])) / (torch.sqrt(v / (1 - _BETAS[1])) + _EPS) + _WD * t["p"])
        return [avg, norm.reshape(1), p, m, v]
    leaves = [t[n].requires_grad_(True) for n in ("w1", "b1", "w2", "b2")]
    w1, b1, w2, b2 = leaves
    loss = ((_gelu(t["x"] @ w1 + b1) @ w2 + b2 - t["t"]) ** 2).mean()
    return [loss.detach(), *torch.autograd.grad(loss, leaves)]
