"""The work that a program gives this framework, as cases that can be timed and checked.

Each case goes through the public entry points (``pratchya_amd.qarr``,
``pratchya_amd.optim``) as a model's code calls them: the quantized Linear
``(QArrayImpl(x, (1, blk)) @ kernel).astype(x.dtype)`` with its two backward
modes, the activation quantizer, the embedding lookup, the output head, the
optimizer's step and the linears of a whole block.
"""
from __future__ import annotations

import math

import torch

from pratchya_amd import optim as O
from pratchya_amd import qarr as Q

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # one generation step of a projection: a few tokens against a weight that stays quantized
        {"name": "decode", "kind": "forward", "rows": 4, "k": 4096, "n": 4096, "blk": 128, "dtype": "bf16"},
        # a prompt of ordinary length through a projection, sizes that no tile divides
        {"name": "prompt ragged", "kind": "forward", "rows": 1000, "k": 2176, "n": 2944, "blk": 128, "dtype": "bf16"},
        # a long batch through the up-projection of a 2048-wide model
        {"name": "forward", "kind": "forward", "rows": 16384, "k": 2048, "n": 8192, "blk": 128, "dtype": "bf16"},
        # the block size 32 preset's projection over a batch
        {"name": "forward blk32", "kind": "forward", "rows": 8192, "k": 4096, "n": 4096, "blk": 32, "dtype": "bf16"},
        # a training step of one Linear with the default backward
        {"name": "train", "kind": "train", "rows": 4096, "k": 2048, "n": 8192, "blk": 128, "dtype": "bf16",
         "backward": "f32"},
        # the same with the block size 16 presets
        {"name": "train blk16", "kind": "train", "rows": 4096, "k": 2048, "n": 2048, "blk": 16, "dtype": "bf16",
         "backward": "f32"},
        # a training step of one Linear with the FP8 backward
        {"name": "train fp8", "kind": "train", "rows": 16384, "k": 2048, "n": 8192, "blk": 128, "dtype": "bf16",
         "backward": "fp8"},
        # an activation into its stored form and back
        {"name": "round trip", "kind": "quantize", "rows": 16384, "k": 2048, "a": 1, "b": 128, "dtype": "bf16"},
        # the rows of a batch's tokens out of the embedding table
        {"name": "embedding", "kind": "embedding", "rows": 8192, "vocab": 65536, "k": 2048, "blk": 128},
        # a batch's logits: the output head's weight has one-column blocks
        {"name": "head", "kind": "head", "rows": 2048, "k": 2048, "n": 32768, "blk": 128},
        # one optimizer step over a layer's weights: stacked bf16 leaves, a 2-D f32 leaf, an embedding, a norm
        {"name": "optimizer", "kind": "optimizer", "layers": 2, "d": 1024, "f": 4096, "blk": 128},
        # the six linears of a 4096-wide block, forward and FP8 backward
        {"name": "block", "kind": "block", "rows": 8192, "d": 4096, "f": 16384, "blk": 128, "backward": "fp8"},
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _side(rng, lo, hi, step=128):
    return max(lo, _between(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(["decode", "prompt", "prompt", "forward", "train", "train", "train fp8", "quantize", "embedding",
                       "head", "optimizer", "block"])
    blk = rng.choice([128, 128, 32, 16])
    if kind == "decode":
        return {"kind": "forward", "rows": _between(rng, 1, 64), "k": _side(rng, 1024, 4096), "n": _side(rng, 1024, 8192),
                "blk": 128, "dtype": "bf16"}
    if kind == "prompt":
        return {"kind": "forward", "rows": _between(rng, 65, 4096), "k": _side(rng, 512, 4096),
                "n": _side(rng, 512, 8192), "blk": blk, "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "forward":
        return {"kind": "forward", "rows": _between(rng, 4096, 16384), "k": 1024 * rng.randint(1, 4),
                "n": 1024 * rng.randint(1, 8), "blk": blk, "dtype": "bf16"}
    if kind == "train":
        return {"kind": "train", "rows": _between(rng, 256, 6144), "k": _side(rng, 512, 2048), "n": _side(rng, 512, 4096),
                "blk": blk, "dtype": rng.choice(["bf16", "bf16", "f32"]), "backward": "f32"}
    if kind == "train fp8":
        return {"kind": "train", "rows": 128 * _between(rng, 4, 128), "k": _side(rng, 512, 4096),
                "n": _side(rng, 512, 8192), "blk": 128, "dtype": "bf16", "backward": "fp8"}
    if kind == "quantize":
        a, b = rng.choice([(1, 128), (1, 32), (1, 16), (128, 128), (32, 32), (16, 16), (128, 1)])
        return {"kind": "quantize", "rows": _between(rng, 1, 128) * 128, "k": _side(rng, 512, 8192), "a": a, "b": b,
                "dtype": rng.choice(["bf16", "f32"])}
    if kind == "embedding":
        return {"kind": "embedding", "rows": _between(rng, 1, 16384), "vocab": _side(rng, 1024, 65536),
                "k": _side(rng, 512, 4096), "blk": blk}
    if kind == "head":
        return {"kind": "head", "rows": _between(rng, 1, 2048), "k": _side(rng, 512, 2048), "n": _side(rng, 4096, 32768),
                "blk": 128}
    if kind == "optimizer":
        return {"kind": "optimizer", "layers": rng.randint(1, 3), "d": _side(rng, 256, 1024), "f": _side(rng, 512, 4096),
                "blk": rng.choice([128, 128, 32])}
    return {"kind": "block", "rows": 128 * _between(rng, 2, 32), "d": _side(rng, 512, 2048), "f": _side(rng, 1024, 8192),
            "blk": 128, "backward": rng.choice(["f32", "fp8"])}


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _activation(gen, rows, k, dtype):
    """N(0, 1) with 1% of the channels 50 times larger, as transformer activations have them."""
    big = torch.where(torch.rand((1, k), generator=gen, device=DEV) < 0.01, 50.0, 1.0)
    return (torch.randn((rows, k), generator=gen, device=DEV) * big).to(dtype)


def _weight(gen, *shape):
    return (torch.randn(shape, generator=gen, device=DEV) * 0.02).to(torch.bfloat16)


def _linears(d, f):
    return [(d, d)] * 4 + [(d, f), (f, d)]


def prepare(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind in ("forward", "head", "train"):
        rows, k, n, blk = case["rows"], case["k"], case["n"], case["blk"]
        s["x"] = _activation(gen, rows, k, DTYPES[case.get("dtype", "bf16")])
        s["w"] = _weight(gen, k, n)
        if kind == "train":
            s["x"].requires_grad_(True)
            s["w"].requires_grad_(True)
            s["g"] = (torch.randn((rows, n), generator=gen, device=DEV) * 1e-3).to(s["x"].dtype)
        else:
            s["wq"] = Q.QArrayImpl(s["w"], (blk, blk if kind == "forward" else 1))
    elif kind == "quantize":
        s["x"] = _activation(gen, case["rows"], case["k"], DTYPES[case["dtype"]])
    elif kind == "embedding":
        s["table"] = Q.QArrayImpl(_weight(gen, case["vocab"], case["k"]), (case["blk"], case["blk"]))
        s["ids"] = torch.randint(0, case["vocab"], (case["rows"],), generator=gen, device=DEV)
    elif kind == "optimizer":
        layers, d, f, grid = case["layers"], case["d"], case["f"], (case["blk"], case["blk"])
        shapes = {"up": (layers, d, f), "down": (layers, f, d), "state": (d, d), "embed_tokens": (2 * f, d)}
        s["params"] = {n: Q.QArrayImpl(_weight(gen, *sh), grid) for n, sh in shapes.items()}
        s["params"]["norm"] = torch.ones(d, device=DEV)
        s["grads"] = {n: (torch.randn(sh, generator=gen, device=DEV) * 1e-3).to(torch.bfloat16)
                      for n, sh in shapes.items()}
        s["grads"]["norm"] = torch.randn(d, generator=gen, device=DEV) * 1e-3
        s["tx"] = O.miulion_optimizer(O.MiulionHyperParams(), O.MiulionScheduler(lambda t: 0.02, lambda t: 3e-4, 0.1))
        # the state after some steps: a momentum that is not zero
        momentum = {n: Q.QArrayImpl(torch.randn(sh, generator=gen, device=DEV) * 1e-3, grid) for n, sh in shapes.items()}
        momentum["norm"] = torch.randn(d, generator=gen, device=DEV) * 1e-3
        s["state"] = O.MiulionState(count=torch.ones([], dtype=torch.int32, device=DEV), momentum=momentum)
    else:
        rows, blk = case["rows"], case["blk"]
        s["xs"], s["ws"], s["gs"] = [], [], []
        for k, n in _linears(case["d"], case["f"]):
            s["xs"].append(_activation(gen, rows, k, torch.bfloat16).requires_grad_(True))
            s["ws"].append(_weight(gen, k, n).requires_grad_(True))
            s["gs"].append((torch.randn((rows, n), generator=gen, device=DEV) * 1e-3).to(torch.bfloat16))
    return s


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------
def _train(x, w, g, blk):
    """Forward and backward of one Linear whose weight an optimizer step has just changed."""
    wq = Q.QArrayImpl(w, (blk, blk))
    y = (Q.QArrayImpl(x, (1, blk)) @ wq).astype(x.dtype)
    gx, gw = torch.autograd.grad(y, (x, w), g)
    return y.detach(), gx, gw


def _bytes(q):
    """A quantized array's stored form."""
    v, s8, s32 = q._tree_flatten()[0]
    return v.view(torch.uint8), s8.view(torch.uint8), s32


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("forward", "head"):
        x = state["x"]
        with torch.no_grad():
            return (Q.QArrayImpl(x, (1, case["blk"])) @ state["wq"]).astype(x.dtype)
    if kind == "train":
        Q.set_matmul_backward(case["backward"])
        return _train(state["x"], state["w"], state["g"], case["blk"])
    if kind == "quantize":
        q = Q.QArrayImpl(state["x"], (case["a"], case["b"]))
        return _bytes(q) + (q.astype(state["x"].dtype),)
    if kind == "embedding":
        return _bytes(state["table"][state["ids"]])
    if kind == "optimizer":
        updates, new = state["tx"].update(state["grads"], state["state"], state["params"])
        names = sorted(updates)
        return ([updates[n] for n in names],
                [_bytes(m) if isinstance(m, Q.QArrayImpl) else m for m in (new.momentum[n] for n in names)])
    Q.set_matmul_backward(case["backward"])
    return [_train(x, w, g, case["blk"]) for x, w, g in zip(state["xs"], state["ws"], state["gs"])]


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def _scales(rows, k, a, b):
    blocks = (rows // a) * (k // b)
    return blocks + 4 * (blocks // math.gcd(max(1, a * b // 16), blocks))


def _train_work(rows, k, n, e):
    return e * (2 * rows * k + 2 * rows * n) + 2 * 2 * k * n, 6 * rows * k * n


def work(case):
    kind = case["kind"]
    e = 4 if case.get("dtype") == "f32" else 2
    if kind in ("forward", "head"):
        rows, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": e * rows * (k + n) + k * n + _scales(k, n, case["blk"], case["blk"] if kind == "forward" else 1),
                "flops": 2 * rows * k * n}
    if kind == "train":
        b, f = _train_work(case["rows"], case["k"], case["n"], e)
        return {"bytes": b, "flops": f}
    if kind == "quantize":
        rows, k = case["rows"], case["k"]
        return {"bytes": rows * k * (2 * e + 1) + _scales(rows, k, case["a"], case["b"]), "flops": 0}
    if kind == "embedding":
        rows, k = case["rows"], case["k"]
        blk = (math.gcd(case["blk"], rows), math.gcd(case["blk"], k))
        return {"bytes": 2 * rows * k + 8 * rows + _scales(rows, k, *blk), "flops": 0}
    if kind == "optimizer":
        layers, d, f = case["layers"], case["d"], case["f"]
        stacked, flat, embed = 2 * layers * d * f, d * d, 2 * f * d
        m = min(d, f)
        # momentum in and out, parameter, gradient and update; five steps of two products (2-D leaves and slices)
        return {"bytes": stacked * (1 + 1 + 1 + 2 + 2) + (flat + embed) * (1 + 1 + 1 + 2 + 4),
                "flops": 5 * 4 * (2 * layers * m * d * f + d * d * d)}
    parts = [_train_work(case["rows"], k, n, 2) for k, n in _linears(case["d"], case["f"])]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    """About four times what the products' rounding was seen to change, against 64 bits.  A product's last
    bits decide e4m3 roundings (steps of 1/8 of a value) of its stored form, and with 128-wide blocks, whose
    products run on FP8 matrix instructions, power-of-two block scales too: such a scale doubles its block's
    cotangent in the reference's backward, which the gradients of a training step show."""
    kind, blk = case["kind"], case.get("blk")
    if kind in ("quantize", "embedding"):
        return "exact"                                      # the stored bytes and what they stand for
    if kind == "head":
        return {"rel": 0.007, "max": 0.016}                 # one bf16 rounding
    if kind == "optimizer":
        return {"rel": 0.025, "max": 0.12}                  # bf16 iterates; the stored momentum is the same bytes
    if kind == "forward":
        if blk != 128:                                      # products to f32 accuracy
            return {"rel": 0.007 if case["dtype"] == "bf16" else 6e-4, "max": 0.5}
        return {"rel": 0.011, "max": 0.5}
    if blk != 128:
        return {"rel": 0.008, "max": 0.5}
    return {"rel": 0.03, "max": 0.99}


# --------------------------------------------------------------------------
# the same in 64 bits, with plain torch
# --------------------------------------------------------------------------
def _blocks(x, a, b):
    h, w = x.shape
    return x.view(h // a, a, w // b, b)


def _quantized(x, grid):
    """(payload, block scale / 128) of a 2-D x in 64 bits; the quantizer is
    defined on 32-bit values, bf16 and e4m3 roundings."""
    a, b = grid
    x = x.detach().float()
    m = _blocks(x, a, b).abs().amax(dim=(1, 3))
    n = m.numel()
    k = math.gcd(max(1, a * b // 16), n)
    top = m.reshape(-1, k).amax(dim=1, keepdim=True)
    r = m.reshape(-1, k) / torch.where(top == 0, 1.0, top)
    s = torch.where(r >= 2.0 ** -126, torch.exp2(torch.frexp(r)[1].double() - 1), 0.0)
    s = (s * top.double()).reshape(m.shape)
    up = lambda v: v[:, None, :, None]   # noqa: E731
    q = (_blocks(x, a, b) / up(s.float().clamp(min=1e-7)) * 128).to(torch.bfloat16).to(torch.float8_e4m3fn)
    return q.reshape(x.shape).double(), s / 128


def _scaled(v, scale, grid):
    """v (64 bits) times its blocks' scales."""
    return (_blocks(v, *grid) * scale[:, None, :, None]).reshape(v.shape)


def _rounded(x, grid):
    """x through its stored form, in 64 bits."""
    q, s = _quantized(x, grid)
    return _scaled(q, s, grid)


def _exact_linear(x, w, gx, gw):
    """(y in 64 bits, its block scales, dequantized x and w)"""
    xd, wd = _rounded(x, gx), _rounded(w, gw)
    go = (gx[0], gw[1])
    q, s = _quantized((xd @ wd).float(), go)
    return _scaled(q, s, go), s, xd, wd


def _exact_train(x, w, g, blk, backward):
    gx, gw, go = (1, blk), (blk, blk), (1, blk)
    y, s, xd, wd = _exact_linear(x, w, gx, gw)
    g1 = _scaled(g.double(), s, go).to(g.dtype)          # the cotangent stays in its own type
    if backward == "f32":
        ga = gb = g1.double()
    else:
        ga, gb, xd = _rounded(g1, (1, 128)), _rounded(g1, (128, 1)), _rounded(xd.float(), (128, 1))
    return y, _rounded((ga @ wd.T).float(), gx), _rounded((xd.T @ gb).float(), gw)


def _exact_direction(c):
    """Five Newton-Schulz steps on c / ||c||."""
    x = c / (c.norm() + 1e-7)
    tall = x.shape[0] > x.shape[1]
    x = x.T if tall else x
    for _ in range(5):
        x = 1.5 * x - 0.5 * (x @ x.T) @ x
    return x.T if tall else x


def _value(q):
    """A quantized array's values in 64 bits, from its stored form."""
    v, s8, s32 = q._tree_flatten()[0]
    grid = q.tgrid
    flat = v.reshape(-1, *v.shape[-2:])
    s8, s32 = s8.reshape(flat.shape[0], -1, s8.shape[-1]), s32.reshape(flat.shape[0], -1, 1)
    out = []
    for i in range(flat.shape[0]):
        s = torch.exp2(s8[i].view(torch.uint8).double() - 127) * s32[i].double() / 128
        out.append(_scaled(flat[i].double(), s.reshape(v.shape[-2] // grid[0], v.shape[-1] // grid[1]), grid))
    return torch.stack(out).reshape(v.shape)


def _exact_optimizer(s):
    updates, momentum = [], []
    for n in sorted(s["params"]):
        p, m, g = s["params"][n], s["state"].momentum[n], s["grads"][n].double()
        quantized = isinstance(p, Q.QArrayImpl)
        p, m = (_value(p), _value(m)) if quantized else (p.double(), m.double())
        c = 0.9 * m + 0.1 * g
        if n in ("embed_tokens", "norm"):
            u, lr = c.sign(), 3e-4
        else:
            u = torch.stack([_exact_direction(v) for v in c.reshape(-1, *c.shape[-2:])]).reshape(c.shape)
            u, lr = u * math.sqrt(max(c.shape[-2:])), 0.02
        updates.append(-(lr * u + lr * 0.1 * p))
        momentum.append((None, None, None) if quantized else 0.99 * m + 0.01 * g)
    return updates, momentum


def exact(case, seed):
    kind = case["kind"]
    if kind == "embedding":
        return None                                       # bytes out of bytes
    s = prepare(case, seed)
    if kind in ("forward", "head"):
        blk = case["blk"]
        return _exact_linear(s["x"], s["w"], (1, blk), (blk, blk if kind == "forward" else 1))[0]
    if kind == "train":
        return _exact_train(s["x"], s["w"], s["g"], case["blk"], case["backward"])
    if kind == "quantize":
        return None, None, None, _rounded(s["x"], (case["a"], case["b"]))
    if kind == "optimizer":
        return _exact_optimizer(s)
    return [_exact_train(x, w, g, case["blk"], case["backward"]) for x, w, g in zip(s["xs"], s["ws"], s["gs"])]
