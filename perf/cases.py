"""The work that users of tbf16 have it do, as cases that can be timed and compared.

A case is a dict of plain values; `prepare` makes what a program has in hand before
the call, `run` is one pass through the public entry points, `exact` the same
results in 64-bit torch, `work` the bytes and operations a pass cannot do without.

Kinds:
  linear           tbf16.scaled_linear on a weight prepared once (inference)
  attention        tbf16.sdpa (inference)
  train_linear     tbf16.autograd.linear and its gradients
  train_attention  tbf16.autograd.sdpa and its gradients
  conv             a converted nn.Conv2d (tbf16.conv.convert_conv), inference
"""
import math
import os
import sys

import torch
import torch.nn as nn

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "turing-bf16_amd"))

import tbf16  # noqa: E402
from tbf16.conv import convert_conv  # noqa: E402

DEV = "cuda"


def listed():
    return [
        # one token of a decoding loop through an MLP up-projection: the smallest call
        {"name": "decode_1", "kind": "linear", "M": 1, "K": 2560, "N": 10240, "bias": False},
        # sixteen sequences decoding together through the same layer
        {"name": "decode_16", "kind": "linear", "M": 16, "K": 2560, "N": 10240, "bias": False},
        # a short prompt through a square projection, outlier rows beyond fp16's range
        {"name": "linear_256", "kind": "linear", "M": 256, "K": 4096, "N": 4096, "bias": False},
        # a vocabulary head with an odd number of tokens
        {"name": "head_odd", "kind": "linear", "M": 100, "K": 1024, "N": 32001, "bias": False},
        # a large projection at prefill
        {"name": "linear_4096", "kind": "linear", "M": 4096, "K": 4096, "N": 4096, "bias": False},
        # causal prefill at an ordinary and at a long context
        {"name": "attention_4k", "kind": "attention", "B": 1, "H": 16, "Hkv": 16, "Sq": 4096, "Sk": 4096, "D": 128,
         "causal": True, "mask": False},
        {"name": "attention_16k", "kind": "attention", "B": 1, "H": 16, "Hkv": 16, "Sq": 16384, "Sk": 16384, "D": 128,
         "causal": True, "mask": False},
        # an encoder's padded batch: ragged length, key-padding mask
        {"name": "attention_mask", "kind": "attention", "B": 2, "H": 12, "Hkv": 12, "Sq": 1111, "Sk": 1111, "D": 64,
         "causal": False, "mask": True},
        # one layer of a training step: a large projection, and a small ragged one with a bias
        {"name": "train_linear", "kind": "train_linear", "M": 8192, "K": 2048, "N": 6144, "bias": False},
        {"name": "train_linear_bias", "kind": "train_linear", "M": 1000, "K": 768, "N": 3072, "bias": True},
        # one attention layer of a training step
        {"name": "train_attention", "kind": "train_attention", "B": 2, "H": 16, "Hkv": 16, "S": 4096, "D": 128,
         "causal": True},
        # a 3x3 convolution of an image decoder
        {"name": "conv_3x3", "kind": "conv", "B": 1, "C": 512, "O": 512, "side": 128, "channels_last": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: mostly a multiple of 64, sometimes only of 8."""
    m = rng.choice((64, 64, 64, 8))
    return max(lo, _log(rng, lo, hi) // m * m)


def draw(rng):
    while True:
        kind = rng.choice(("linear",) * 4 + ("attention",) * 2 + ("train_linear",) * 2 + ("train_attention", "conv"))
        if kind == "linear":
            c = {"kind": kind, "M": _log(rng, 1, 8192), "K": _width(rng, 256, 8192), "N": _width(rng, 256, 16384),
                 "bias": rng.random() < 0.5}
            if rng.random() < 0.15:
                c["N"] += rng.randrange(1, 8)
            if 2 * c["M"] * c["K"] * c["N"] <= 2.8e11 and c["K"] * c["N"] <= 1 << 26:
                return c
        elif kind == "attention":
            causal = rng.random() < 0.5
            Sq = _log(rng, 32, 16384)
            Sk = Sq if causal or rng.random() < 0.5 else _log(rng, 32, 8192)
            Hkv = rng.choice((2, 4, 8, 12, 16))
            c = {"kind": kind, "B": rng.choice((1, 1, 2, 4)), "H": Hkv * rng.choice((1, 1, 1, 4)), "Hkv": Hkv, "Sq": Sq,
                 "Sk": Sk, "D": rng.choice((64, 64, 80, 96, 128, 128, 128)), "causal": causal,
                 "mask": not causal and rng.random() < 0.4}
            if work(c)["flops"] <= 1.1e12 and c["H"] <= 32:
                return c
        elif kind == "train_linear":
            c = {"kind": kind, "M": _log(rng, 64, 8192), "K": _width(rng, 256, 4096), "N": _width(rng, 256, 8192),
                 "bias": rng.random() < 0.5}
            if work(c)["flops"] <= 6.2e11:
                return c
        elif kind == "train_attention":
            Hkv = rng.choice((4, 8, 12, 16))
            c = {"kind": kind, "B": rng.choice((1, 2, 4)), "H": Hkv * rng.choice((1, 1, 2)), "Hkv": Hkv,
                 "S": _log(rng, 64, 4096), "D": rng.choice((64, 64, 96, 128, 128)), "causal": rng.random() < 0.6}
            if work(c)["flops"] <= 4.9e11:
                return c
        else:
            c = {"kind": kind, "B": rng.choice((1, 2)), "C": 32 * rng.randrange(2, 17), "O": 32 * rng.randrange(2, 17),
                 "side": _log(rng, 16, 128), "channels_last": rng.random() < 0.5}
            if work(c)["flops"] <= 8e10:
                return c


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _rows(g, M, K):
    """Activations: N(0, 1) rows, one in twenty an outlier token beyond fp16's range."""
    x = _randn(g, M, K)
    big = torch.rand(M, generator=g, device=DEV) < 0.05
    return (x * torch.where(big, 2.0 ** 17, 1.0)[:, None]).bfloat16()


def _heads(g, B, H, S, D, lo, hi):
    """N(0, 1) heads, each scaled by 2^u with u uniform in [lo, hi]."""
    u = lo + (hi - lo) * torch.rand(B, H, 1, 1, generator=g, device=DEV)
    return (_randn(g, B, H, S, D) * torch.exp2(u)).bfloat16()


def _inputs(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("linear", "train_linear"):
        M, K, N = case["M"], case["K"], case["N"]
        s = {"x": _rows(g, M, K), "w": (_randn(g, N, K) * K ** -0.5).bfloat16(),
             "b": _randn(g, N).bfloat16() if case["bias"] else None}
        if kind == "train_linear":
            s["dy"] = (_randn(g, M, N) * 1e-3).bfloat16()
        return s
    if kind == "attention":
        B, H, Hkv, Sq, Sk, D = (case[n] for n in ("B", "H", "Hkv", "Sq", "Sk", "D"))
        s = {"q": _heads(g, B, H, Sq, D, 0.0, 2.0), "k": _heads(g, B, Hkv, Sk, D, 0.0, 2.0),
             "v": _heads(g, B, Hkv, Sk, D, -4.0, 12.0), "mask": None}
        if case["mask"]:
            length = torch.randint(Sk // 2 + 1, Sk + 1, (B, 1, 1, 1), generator=g, device=DEV)
            s["mask"] = torch.arange(Sk, device=DEV).view(1, 1, 1, Sk) < length
        return s
    if kind == "train_attention":
        B, H, Hkv, S, D = (case[n] for n in ("B", "H", "Hkv", "S", "D"))
        return {"q": _randn(g, B, H, S, D).bfloat16(), "k": _randn(g, B, Hkv, S, D).bfloat16(),
                "v": _randn(g, B, Hkv, S, D).bfloat16(), "do": (_randn(g, B, H, S, D) * 2.0 ** -20).bfloat16()}
    B, C, O, side = (case[n] for n in ("B", "C", "O", "side"))
    return {"x": (_randn(g, B, C, side, side) * 2.0 ** 10).bfloat16(),
            "w": (_randn(g, O, C, 3, 3) * (9 * C) ** -0.5).bfloat16(), "b": _randn(g, O).bfloat16()}


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["kind"] == "linear":
        s["w16"], s["ws"] = tbf16.prepare_weight(s.pop("w"))  # once per weight, kept by the program
    elif case["kind"] == "conv":
        conv = nn.Conv2d(case["C"], case["O"], 3, padding=1, device=DEV, dtype=torch.bfloat16)
        with torch.no_grad():
            conv.weight.copy_(s.pop("w"))
            conv.bias.copy_(s.pop("b"))
        if case["channels_last"]:
            conv = conv.to(memory_format=torch.channels_last)
            s["x"] = s["x"].to(memory_format=torch.channels_last)
        s["conv"] = convert_conv(conv)
    return s


def _leaf(t):
    """A new leaf on the same storage: each pass sees its activations as new tensors."""
    return t.detach().requires_grad_()


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return tbf16.scaled_linear(state["x"], state["w16"], state["ws"], state["b"])
    if kind == "attention":
        return tbf16.sdpa(state["q"], state["k"], state["v"], attn_mask=state["mask"], is_causal=case["causal"],
                          enable_gqa=case["H"] != case["Hkv"])
    if kind == "train_linear":
        leaves = [_leaf(state[n]) for n in ("x", "w", "b") if state[n] is not None]
        y = tbf16.autograd.linear(*leaves)
        return (y.detach(), *torch.autograd.grad(y, leaves, state["dy"]))
    if kind == "train_attention":
        leaves = [_leaf(state[n]) for n in ("q", "k", "v")]
        o = tbf16.autograd.sdpa(*leaves, is_causal=case["causal"], enable_gqa=case["H"] != case["Hkv"])
        return (o.detach(), *torch.autograd.grad(o, leaves, state["do"]))
    with torch.no_grad():
        return state["conv"](state["x"])


def work(case):
    kind = case["kind"]
    if kind in ("linear", "train_linear"):
        M, K, N = case["M"], case["K"], case["N"]
        b = 2 * N if case["bias"] else 0
        if kind == "linear":
            return {"bytes": 2 * (M * K + N * K + M * N) + 4 * N + b, "flops": 2 * M * K * N}
        return {"bytes": 2 * (2 * M * K + 2 * N * K + 2 * M * N) + 2 * b, "flops": 6 * M * K * N}
    if kind == "attention":
        B, H, Hkv, Sq, Sk, D = (case[n] for n in ("B", "H", "Hkv", "Sq", "Sk", "D"))
        return {"bytes": 2 * B * D * (2 * H * Sq + 2 * Hkv * Sk) + (B * Sk if case["mask"] else 0),
                "flops": (2 if case["causal"] else 4) * B * H * Sq * Sk * D}
    if kind == "train_attention":
        B, H, Hkv, S, D = (case[n] for n in ("B", "H", "Hkv", "S", "D"))
        return {"bytes": 2 * B * D * S * (4 * H + 4 * Hkv), "flops": (7 if case["causal"] else 14) * B * H * S * S * D}
    B, C, O, side = (case[n] for n in ("B", "C", "O", "side"))
    P = B * side * side
    return {"bytes": 2 * (P * C + P * O + 9 * C * O + O), "flops": 18 * P * C * O}


def tolerance(case):
    # bf16 results of fp32 sums are 1.4e-3 to 1.7e-3 off the 64-bit ones by their rounding;
    # four times that
    return {"rel": 7e-3}


def _attention64(q, k, v, causal, mask, do=None):
    """(o,) or (o, dq, dk, dv) of one head in 64 bits; q is (Sq, D), mask (Sk,) or None."""
    scale = q.shape[-1] ** -0.5
    s = (q @ k.t()) * scale
    if causal:
        s.masked_fill_(torch.ones_like(s, dtype=torch.bool).triu_(1), -math.inf)
    if mask is not None:
        s.masked_fill_(~mask, -math.inf)
    p = torch.softmax(s, -1)
    del s
    o = p @ v
    if do is None:
        return (o,)
    ds = p * (do @ v.t() - (do * o).sum(-1, keepdim=True)) * scale
    return o, ds @ k, ds.t() @ q, p.t() @ do


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("linear", "train_linear"):
        x, w = s["x"].double(), s["w"].double()
        y = x @ w.t()
        if s["b"] is not None:
            y += s["b"].double()
        if kind == "linear":
            return y
        dy = s["dy"].double()
        return (y, dy @ w, dy.t() @ x) + ((dy.sum(0),) if s["b"] is not None else ())
    if kind in ("attention", "train_attention"):
        train = kind == "train_attention"
        q, k, v = s["q"], s["k"], s["v"]
        B, H = q.shape[:2]
        group = H // k.shape[1]
        outs = [torch.zeros(t.shape, dtype=torch.float64, device=DEV) for t in ((q, q, k, v) if train else (q,))]
        for b in range(B):
            mask = s["mask"][b, 0, 0] if s.get("mask") is not None else None
            for h in range(H):
                got = _attention64(q[b, h].double(), k[b, h // group].double(), v[b, h // group].double(),
                                   case["causal"], mask, s["do"][b, h].double() if train else None)
                for i, (o, t) in enumerate(zip(outs, got)):
                    o[b, h if i < 2 else h // group] += t
        return tuple(outs) if train else outs[0]
    x, w = s["x"].double(), s["w"].double()
    B, C, O, side = (case[n] for n in ("B", "C", "O", "side"))
    xp = torch.nn.functional.pad(x, (1, 1, 1, 1))
    y = s["b"].double()[:, None].expand(O, side * side).repeat(B, 1, 1)
    for b in range(B):
        for i in range(3):
            for j in range(3):
                y[b] += w[:, :, i, j] @ xp[b, :, i:i + side, j:j + side].reshape(C, side * side)
    y = y.reshape(B, O, side, side)
    return y.to(memory_format=torch.channels_last) if case["channels_last"] else y
