"""Timed workloads of the fused attention operators, called as a user's program calls them.

A case is one call pattern: the entry point and operand layout ("path"), the sizes, the mask, and
whether only the forward runs (inference) or the forward and the backward (training). Paths:
  qkv      fused_attention_qkv on the [b, s, 3 h d] output of a fused projection;
  views    fused_attention on the three head-split views of such a projection;
  strided  fused_attention on transpose(1, 2) views of three [b, s, h, d] buffers (the outputs of
           three separate projections);
  general  fused_attention on three contiguous [b, h, s, d] tensors.
Inputs are N(0, std^2), the output gradient N(0, 1), scale 1 / sqrt(d). Everything is fp32: the
operators take no other type.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = Path(__file__).resolve().parent.parent / "candle-fused-attn_amd"
if str(_PKG) not in sys.path:
    sys.path.insert(0, str(_PKG))

import candle_fused_attn as cfa  # noqa: E402

PATHS = ("qkv", "views", "strided", "general")
DEVICE = "cuda:0"


def _case(name, path, b, h, s, d, causal, train, std=1.0):
    return {"name": name, "path": path, "b": b, "h": h, "s": s, "d": d, "causal": causal,
            "train": train, "std": std}


def listed():
    return [
        # One short prompt through one small layer: launch and host latency are what counts.
        _case("tiny_fwd", "qkv", 1, 2, 33, 64, True, False),
        # The smallest training call of the benchmark configurations: separate q, k, v tensors.
        _case("small_train", "general", 2, 4, 128, 64, False, True),
        # The headline shape (an encoder layer over 240 tokens), inference.
        _case("encoder_fwd", "qkv", 64, 6, 240, 64, False, False),
        # The headline shape, a training step.
        _case("encoder_train", "qkv", 64, 6, 240, 64, False, True),
        # The same, causal (a small decoder).
        _case("decoder_train", "qkv", 64, 6, 240, 64, True, True),
        # A long-context decoder layer's training step.
        _case("long_decoder_train", "qkv", 8, 12, 2048, 64, True, True),
        # Separate projections read in place, large logits, an encoder over 1024 tokens.
        _case("strided_train", "strided", 16, 16, 1024, 64, False, True, 2.0),
        # Narrow heads.
        _case("d32_train", "qkv", 64, 6, 240, 32, False, True),
        # Wide heads.
        _case("d128_train", "views", 64, 6, 240, 128, False, True),
        # The prefill of one long prompt, wide heads: few (batch, head) pairs.
        _case("d128_prefill", "qkv", 1, 16, 4096, 128, True, False),
        # A ragged batch: odd sizes everywhere, head views of one projection.
        _case("ragged_train", "views", 3, 5, 333, 64, False, True),
        # An odd mid-size decoder step on separate contiguous tensors.
        _case("odd_decoder_train", "general", 4, 9, 777, 64, True, True),
    ]


# The most a drawn case may cost: the listed strided_train's.
_MAX_FLOPS = 14 * 64 * 16 * 16 * 1024 * 1024
_MAX_ROWS = 16 * 16 * 1024 * 64  # b h s d


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    d = rng.choice((32, 64, 64, 64, 128))
    causal, train = rng.random() < 0.5, rng.random() < 0.7
    s = _log_uniform(rng, 16, 4096)
    if rng.random() < 0.5 and s > 16:
        s |= 1  # odd lengths as often as not
    most = int(min(1024, _MAX_FLOPS / (14 * d * s * s), _MAX_ROWS / (s * d)))
    pairs = _log_uniform(rng, 1, max(most, 1))
    h = min(pairs, rng.choice((1, 2, 3, 5, 6, 8, 12, 16)))
    return {"path": rng.choice(PATHS), "b": max(pairs // h, 1), "h": h, "s": s, "d": d,
            "causal": causal, "train": train, "std": rng.choice((1.0, 1.0, 2.0))}


def _inputs(case, seed):
    """The operand leaves and the output gradient [b, s, h, d], made on the GPU from the seed."""
    b, h, s, d = case["b"], case["h"], case["s"], case["d"]
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)

    def normal(*shape, std=1.0):
        return torch.randn(*shape, generator=gen, device=DEVICE, dtype=torch.float32) * std

    if case["path"] in ("qkv", "views"):
        leaves = [normal(b, s, 3 * h * d, std=case["std"])]
    elif case["path"] == "strided":
        leaves = [normal(b, s, h, d, std=case["std"]) for _ in range(3)]
    else:
        leaves = [normal(b, h, s, d, std=case["std"]) for _ in range(3)]
    return leaves, normal(b, s, h, d)


def prepare(case, seed):
    leaves, grad = _inputs(case, seed)
    if case["train"]:
        for t in leaves:
            t.requires_grad_(True)
        if case["path"] == "qkv":
            grad = grad.view(case["b"], case["s"], case["h"] * case["d"])
    else:
        grad = None
    return {"case": case, "leaves": leaves, "grad": grad}


def _attend(case, leaves):
    """The operator's output, heads merged or mergeable: [b, s, h d] (qkv), else [b, s, h, d]."""
    b, h, s, d = case["b"], case["h"], case["s"], case["d"]
    scale, causal = 1.0 / math.sqrt(d), case["causal"]
    if case["path"] == "qkv":
        return cfa.fused_attention_qkv(leaves[0], h, scale, causal)
    if case["path"] == "views":
        q, k, v = (leaves[0].narrow(2, i * h * d, h * d).view(b, s, h, d).transpose(1, 2)
                   for i in range(3))
    elif case["path"] == "strided":
        q, k, v = (t.transpose(1, 2) for t in leaves)
    else:
        q, k, v = leaves
    return cfa.fused_attention(q, k, v, scale, causal).transpose(1, 2)


def run(state):
    case, leaves = state["case"], state["leaves"]
    if not case["train"]:
        with torch.no_grad():
            return [_attend(case, leaves)]
    out = _attend(case, leaves)
    return [out.detach(), *torch.autograd.grad(out, leaves, state["grad"])]


def _pairs(case):
    """(query, key) pairs that attention has to score."""
    s = case["s"]
    return case["b"] * case["h"] * (s * (s + 1) // 2 if case["causal"] else s * s)


def work(case):
    """Two products forward (4 d per pair), five backward (10 d per pair); q, k, v read and O
    written, and for the backward q, k, v, O and dO read and dQ, dK, dV written."""
    elems = case["b"] * case["h"] * case["s"] * case["d"]
    flops = (14 if case["train"] else 4) * case["d"] * _pairs(case)
    return {"bytes": 4 * elems * (4 + (8 if case["train"] else 0)), "flops": flops}


def tolerance(case):
    """fp32 products and sums in another order: about four times the largest error against fp64
    seen over the listed and a few hundred drawn cases."""
    return {"rel": 3e-6}


def exact(case, seed):
    """Attention and its gradients in float64 by plain torch, (b, h) pairs a few at a time."""
    b, h, s, d = case["b"], case["h"], case["s"], case["d"]
    leaves, grad = _inputs(case, seed)
    if case["path"] in ("qkv", "views"):
        parts = leaves[0].view(b, s, 3, h, d).unbind(2)
        q, k, v = (t.transpose(1, 2) for t in parts)
    elif case["path"] == "strided":
        q, k, v = (t.transpose(1, 2) for t in leaves)
    else:
        q, k, v = leaves
    q, k, v, g = (t.reshape(b * h, s, d) for t in (q, k, v, grad.transpose(1, 2)))
    scale = 1.0 / math.sqrt(d)
    mask = (torch.ones(s, s, dtype=torch.bool, device=DEVICE).triu(1) if case["causal"] else None)
    o, dq, dk, dv = (torch.empty(b * h, s, d, dtype=torch.float64, device=DEVICE)
                     for _ in range(4))
    step = max(1, (1 << 26) // (s * s))
    for i in range(0, b * h, step):
        at = slice(i, i + step)
        qi, ki, vi, gi = (t[at].double() for t in (q, k, v, g))
        p = torch.matmul(qi, ki.transpose(1, 2).contiguous()) * scale
        if mask is not None:
            p.masked_fill_(mask, -math.inf)
        p = torch.softmax(p, dim=-1)
        o[at] = torch.matmul(p, vi)
        if not case["train"]:
            continue
        pt = p.transpose(1, 2).contiguous()
        dv[at] = torch.matmul(pt, gi)
        ds = torch.matmul(gi, vi.transpose(1, 2).contiguous())
        ds -= (gi * o[at]).sum(-1, keepdim=True)
        ds *= p
        ds *= scale
        dq[at] = torch.matmul(ds, ki)
        dk[at] = torch.matmul(ds.transpose(1, 2).contiguous(), qi)

    def to_bshd(t):
        return t.view(b, h, s, d).transpose(1, 2)

    out = to_bshd(o)
    if case["path"] == "qkv":
        out = out.reshape(b, s, h * d)
    if not case["train"]:
        return [out]
    if case["path"] in ("qkv", "views"):
        grads = [torch.stack([to_bshd(t) for t in (dq, dk, dv)], dim=2).reshape(b, s, 3 * h * d)]
    elif case["path"] == "strided":
        grads = [to_bshd(t) for t in (dq, dk, dv)]
    else:
        grads = [t.view(b, h, s, d) for t in (dq, dk, dv)]
    return [out, *grads]
