"""The work this library is asked to do, as cases that can be timed and checked.

Every case is one pass through the public Python mirror of the C ABI
(`demonic_amd`), as a decode or prefill loop calls it.  Weights are
N(0, 0.02) bf16 bit patterns (f32 where the case says so) and activations
N(0, 1) f32, the distributions of the repository's own configurations; shapes
are Llama-3-8B's projections, the repository's edge shapes, and generic ones.

kind      entry point                          a pass is
rd        gemv_rd                              y = x @ W', W [n,k] in a device region
layer     gemv_rd_grouped / gemv_rd            the 7 projections of one transformer layer
cs        gemv_cs                              y[z] = x[z] @ W[z], W [batch,k,n] in a device region
f32       gemv_f32_rd                          y = x @ W', f32 weights in a device region
dropin    matmul_bf16_gpu / _t                 the drop-in `@` on host arrays, weight resident by content
"""
import math

import numpy as np
import torch

import demonic_amd as hip

UP_N, HIDDEN = 14336, 4096          # Llama-3-8B FFN width and model width
MAX_WEIGHT = 128256 * HIDDEN        # elements of the LM head
MAX_MACS = UP_N * HIDDEN * 2048     # multiply-adds of the longest listed prefill


def listed():
    return [
        # one GPU's share of the gate/up projection under 8-way tensor parallelism: the smallest
        # weight a decode step reads alone, a few microseconds, so launches count
        {"name": "share_m1", "kind": "rd", "m": 1, "n": 1792, "k": 4096},
        # one decode token through a layer: q/k/v and gate/up grouped, o and down alone
        {"name": "layer_m1", "kind": "layer", "m": 1, "hidden": HIDDEN, "kv": 1024, "ffn": UP_N},
        # the LM head for a batch of 16 sequences: the largest weight
        {"name": "lm_head_m16", "kind": "rd", "m": 16, "n": 128256, "k": HIDDEN},
        # batched decode / a short prefill: 64 activation rows against gate/up
        {"name": "up_m64", "kind": "rd", "m": 64, "n": UP_N, "k": HIDDEN},
        # prefill chunks of 512 and 2048 tokens against gate/up and down
        {"name": "up_m512", "kind": "rd", "m": 512, "n": UP_N, "k": HIDDEN},
        {"name": "down_m2048", "kind": "rd", "m": 2048, "n": HIDDEN, "k": UP_N},
        # rows of odd length (the edge configuration's shape), one token and a batch
        {"name": "odd_m1", "kind": "rd", "m": 1, "n": 11008, "k": 4097},
        {"name": "odd_m33", "kind": "rd", "m": 33, "n": 11008, "k": 4097},
        # `x @ W` on a weight kept as [k,n] in a device region, the language's own layout: one token
        # and a short prefill
        {"name": "kn_m1", "kind": "cs", "m": 1, "batch": 1, "n": UP_N, "k": HIDDEN, "shared_x": False},
        {"name": "kn_m64", "kind": "cs", "m": 64, "batch": 1, "n": UP_N, "k": HIDDEN, "shared_x": False},
        # f32 weights, a batch of 8
        {"name": "f32_m8", "kind": "f32", "m": 8, "n": UP_N, "k": HIDDEN},
        # the drop-in `x @ W` with host x and y: one synchronous call per `@`
        {"name": "dropin_m1", "kind": "dropin", "m": 1, "n": HIDDEN, "k": HIDDEN, "transposed": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size of [lo, hi], spread over its logarithm: mostly multiples of 64, some of 8, some odd."""
    v, u = _log(rng, lo, hi), rng.random()
    return max(lo, v // 64 * 64) if u < 0.6 else max(lo, v // 8 * 8) if u < 0.75 else v


def _rows(rng, most):
    """Activation rows: decode batches (1..16) and prefill chunks alike."""
    return _log(rng, 1, 16) if most <= 16 or rng.random() < 0.5 else _log(rng, 17, most)


def draw(rng):
    u = rng.random()
    while True:
        if u < 0.5:
            c = {"kind": "rd", "m": _rows(rng, 2048), "n": _size(rng, 512, 131072), "k": _size(rng, 512, 16384)}
        elif u < 0.6:
            h = 256 * _log(rng, 4, 24)
            c = {"kind": "layer", "m": _log(rng, 1, 4), "hidden": h, "kv": h // 4, "ffn": 256 * (h * 7 // 512)}
            return c
        elif u < 0.75:
            c = {"kind": "cs", "m": _rows(rng, 64), "batch": 1, "n": _size(rng, 512, 32768),
                 "k": _size(rng, 512, 16384), "shared_x": False}
            if rng.random() < 0.4:  # per-head projections
                c.update(m=1, batch=rng.randint(4, 32), n=64 * rng.randint(1, 4), shared_x=rng.random() < 0.5)
        elif u < 0.87:
            c = {"kind": "f32", "m": _rows(rng, 16), "n": _size(rng, 512, 32768), "k": _size(rng, 512, 16384)}
        else:
            c = {"kind": "dropin", "m": _rows(rng, 64), "n": _size(rng, 512, 8192), "k": _size(rng, 512, 8192),
                 "transposed": rng.random() < 0.5}
        w = c["n"] * c["k"] * c.get("batch", 1) * (2 if c["kind"] == "f32" else 1)
        if w <= MAX_WEIGHT and w * c["m"] <= MAX_MACS and (c["kind"] != "dropin" or w <= 1 << 25):
            return c


def _problems(case):
    """(weight rows or columns n, k) of each product of a pass, and the activation each one reads."""
    if case["kind"] != "layer":
        return [(case["n"], case["k"], 0)]
    h, kv, f = case["hidden"], case["kv"], case["ffn"]
    return [(h, h, 0), (kv, h, 0), (kv, h, 0), (h, h, 1), (f, h, 2), (f, h, 2), (h, f, 3)]


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def _weight(gen, scale, *shape):
    """bf16 bit patterns of N(0, scale), in pieces so that a large one needs no f32 copy of itself."""
    w = torch.empty(shape, device="cuda", dtype=torch.bfloat16)
    flat = w.view(-1)
    for i in range(0, flat.numel(), 1 << 26):
        piece = flat[i:i + (1 << 26)]
        piece.copy_(_randn(gen, piece.numel()) * scale)
    return w


def _inputs(case, seed):
    """The activations and weights of a case, from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed * 1000003 + 17)
    m, probs, batch = case["m"], _problems(case), case.get("batch", 1)
    xs = {}
    for n, k, i in probs:
        if i not in xs:
            xs[i] = _randn(gen, *((m, k) if batch == 1 or case.get("shared_x") else (batch, m, k)))
    ws = []
    for n, k, i in probs:
        if case["kind"] == "f32":
            ws.append(_randn(gen, n, k) * 0.02)
        elif case["kind"] == "cs":
            ws.append(_weight(gen, 0.02, batch, k, n))
        elif case["kind"] == "dropin" and not case["transposed"]:
            ws.append(_weight(gen, 0.02, k, n))
        else:
            ws.append(_weight(gen, 0.02, n, k))
    return [xs[i] for i in sorted(xs)], ws


def prepare(case, seed):
    xs, ws = _inputs(case, seed)
    if case["kind"] == "dropin":
        return {"case": case, "x": xs[0].cpu().numpy(), "w": ws[0].view(torch.int16).cpu().numpy().view(np.uint16)}
    ys = [torch.empty((case.get("batch", 1), case["m"], n) if case["kind"] == "cs" else (case["m"], n),
                      device="cuda", dtype=torch.float32) for n, _, _ in _problems(case)]
    torch.cuda.synchronize()  # the library runs on its own stream: its inputs are ready before the first call
    return {"case": case, "xs": xs, "ws": ws, "ys": ys,
            "xa": [x.data_ptr() for x in xs], "wa": [w.data_ptr() for w in ws], "ya": [y.data_ptr() for y in ys]}


def run(state):
    c = state["case"]
    kind, m = c["kind"], c["m"]
    if kind == "dropin":
        return (hip.matmul_bf16_gpu_t if c["transposed"] else hip.matmul_bf16_gpu)(state["x"], state["w"])
    x, w, y = state["xa"], state["wa"], state["ya"]
    if kind == "rd":
        hip.gemv_rd(x[0], w[0], y[0], m, c["k"], c["n"])
    elif kind == "cs":
        k, n = c["k"], c["n"]
        hip.gemv_cs(x[0], w[0], y[0], m, k, n, c["batch"], 0 if c["shared_x"] else m * k, k * n)
    elif kind == "f32":
        hip.gemv_f32_rd(x[0], w[0], y[0], m, c["k"], c["n"])
    else:
        h, kv, f = c["hidden"], c["kv"], c["ffn"]
        hip.gemv_rd_grouped([x[0]] * 3, w[:3], y[:3], [h, kv, kv], m, h)
        hip.gemv_rd(x[1], w[3], y[3], m, h, h)
        hip.gemv_rd_grouped([x[2]] * 2, w[4:6], y[4:6], [f, f], m, h)
        hip.gemv_rd(x[3], w[6], y[6], m, f, h)
    return state["ys"]


def work(case):
    m, batch, size = case["m"], case.get("batch", 1), 4 if case["kind"] == "f32" else 2
    macs = sum(n * k for n, k, _ in _problems(case)) * batch
    xs = {i: k for n, k, i in _problems(case)}
    x = sum(xs.values()) * m * (1 if case.get("shared_x") else batch)
    y = sum(n for n, _, _ in _problems(case)) * m * batch
    return {"bytes": size * macs + 4 * x + 4 * y, "flops": 2 * macs * m}


def tolerance(case):
    # f32 sums of up to 16384 products in any order.
    return {"rel": 4e-6}


def exact(case, seed):
    xs, ws = _inputs(case, seed)
    out = []
    for (n, k, i), w in zip(_problems(case), ws):
        x = xs[i].double()
        if case["kind"] == "cs":
            x = x.expand(case["batch"], case["m"], k) if x.dim() == 2 else x
            out.append(torch.stack([x[z] @ w[z].double() for z in range(case["batch"])]))
        elif case["kind"] == "dropin" and not case["transposed"]:
            return (x @ w.double()).cpu().numpy()
        else:  # W [n,k], in blocks of rows
            y = torch.cat([x @ w[r:r + 16384].double().t() for r in range(0, n, 16384)], 1)
            if case["kind"] == "dropin":
                return y.cpu().numpy()
            out.append(y)
    return out
