"""Rows of very different size in one call: what a row of the results loses to a row that has no part
in it, or to a term far larger than its own. Every row is checked against fp64.

The bar: products and sums in fp32 leave a few 1e-7 of the size of a row's terms (REL_TOL, as for
whole results); a weight exp(x) adds |x| 2^-24 for each rounding of its argument, four of which reach
a gradient (x as formed and as subtracted, in the forward's sum and in the backward's weight). For O
and dV, sums of weighted rows, it is relative to the row itself; for dQ and dK, whose terms hold the
difference dP - D, to the row of the terms' magnitudes.
"""
from __future__ import annotations

import math

import pytest
import torch

from test_pair_gpu import REL_TOL, forward, gradients, normal, reference

pytestmark = pytest.mark.gpu


def bar(x):
    return REL_TOL + 4 * abs(x) * 2.0 ** -24


def everything(q, k, v, g, scale, causal):
    """name -> (result, fp64 reference, what its rows' errors are relative to)."""
    want = reference(q, k, v, scale, causal, g)
    got = [forward(q, k, v, scale, causal), *gradients(q, k, v, g, scale, causal)]
    q, k, v, g = (t.double().cpu() for t in (q, k, v, g))
    x = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
    if causal:
        x = x.masked_fill(torch.ones(x.shape[1:], dtype=torch.bool).triu(1), -math.inf)
    p = torch.softmax(x, dim=-1)
    terms = torch.matmul(g.abs(), v.abs().transpose(1, 2).contiguous())
    terms = p * (terms + (g.abs() * torch.matmul(p, v.abs())).sum(-1, keepdim=True)) * scale
    size = [want[0], torch.matmul(terms, k.abs()),
            torch.matmul(terms.transpose(1, 2).contiguous(), q.abs()), want[3]]
    return {n: t for n, *t in zip(("o", "dq", "dk", "dv"), got, want, size)}


def check_rows(name, result, tol, rows=slice(None)):
    """Rows are the second dimension; a row whose terms are all 0 has to be 0."""
    got, want, size = (t.detach().double().cpu()[:, rows] for t in result)
    diff, size = (got - want).norm(dim=-1), size.norm(dim=-1)
    assert torch.isfinite(diff).all(), name
    assert (diff[size == 0] == 0).all(), name
    worst = (diff / size.clamp_min(1e-300)).max().item()
    print(f"{name}: worst row {worst:.2e} (bar {tol:.2e})", flush=True)
    assert worst <= tol, name


def with_logit(q, k, row, logit, scale):
    """Key `row` scores `logit` with every query; the others keep their scores."""
    q[:, :, 0], k[:, :, 0] = 4.0, 0.0
    k[:, row] = 0.0
    k[:, row, 0] = logit / (4.0 * scale)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("logit", [8.0, 14.0, 24.0])
def test_sink(cuda, logit, d, causal):
    """An attention sink: one key takes nearly all weight, its value is (nearly) zero, so that the
    output and the gradients are made by the small weights of the others."""
    s, scale = 2048 if d == 64 else 600, 1.0 / math.sqrt(d)
    for value in (0.0, 1e-3):
        q, k, v, g = (normal(200 + i, 2, s, d) for i in range(4))
        with_logit(q, k, 0, logit, scale)
        v[:, 0] *= value
        for name, r in everything(q, k, v, g, scale, causal).items():
            check_rows(f"sink {logit} value {value} d{d} causal={causal} {name}", r,
                       bar(logit + math.log(s)))


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("power", [12, 24, 60])
def test_large_row_without_weight(cuda, d, power):
    """One row of V, K, Q or dO times 2^power: causal, the queries before it (V, K) and the keys
    after it (Q, dO) have no part in it; not causal, a V row whose weight is 0."""
    s, at, scale = 150, 70, 1.0 / math.sqrt(d)
    x = [normal(220 + i, 2, s, d) for i in range(4)]
    for name, which in (("v", 2), ("k", 1), ("q", 0), ("dO", 3)):
        y = [t.clone() for t in x]
        # (K and Q: scores of +-2^power, a softmax of 0s and 1s where the row has a part.)
        y[which][:, at] *= 2.0 ** power
        q, k, v, g = y
        rows = {"o": slice(0, at), "dq": slice(0, at)}
        if name in ("q", "dO"):
            rows |= {"dk": slice(at + 1, s), "dv": slice(at + 1, s)}
        results = everything(q, k, v, g, scale, True)
        for out, r in rows.items():
            check_rows(f"large {name} 2^{power} d{d} {out}", results[out], bar(8), r)
    q, k, v, g = (t.clone() for t in x)
    with_logit(q, k, at, -400.0, scale)
    v[:, at] *= 2.0 ** power
    check_rows(f"weightless 2^{power} d{d} o", everything(q, k, v, g, scale, False)["o"], bar(8))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("logit", [-12.0, -24.0, -40.0])
def test_rarely_attended_key(cuda, logit, d, causal):
    """A key of small weight with every query: its own dK and dV."""
    s, at, scale = 300, 33, 1.0 / math.sqrt(d)
    for n in (2, 40):  # (causal, either side of the serial dV rule)
        q, k, v, g = (normal(240 + i, n, s, d) for i in range(4))
        with_logit(q, k, at, logit, scale)
        results = everything(q, k, v, g, scale, causal)
        for name in ("dk", "dv"):
            check_rows(f"rare key {logit} d{d} causal={causal} n{n} {name}", results[name],
                       bar(logit - math.log(s)), slice(at, at + 1))


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("grow", [2, 6])
def test_rows_of_every_size(cuda, d, grow):
    """Rows of V and dO of sizes 2^(+-grow ...) in no order: each key's dV and each query's O and dQ
    are sums of terms of very different size."""
    s, scale = 200, 1.0 / math.sqrt(d)
    q, k, v, g = (normal(260 + i, 2, s, d) for i in range(4))
    power = torch.randint(-4, 5, (2, s, 1), generator=torch.Generator().manual_seed(9)).to(q)
    v, g = v * torch.exp2(grow * power), g * torch.exp2(grow * power.roll(7, 1))
    for causal in (False, True):
        for name, r in everything(q, k, v, g, scale, causal).items():
            check_rows(f"sizes {grow} d{d} causal={causal} {name}", r, bar(8))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("logit", [60.0, 76.0])
def test_late_sink(cuda, logit, d, causal):
    """A sink of value zero after tiles of ordinary keys, which its weight makes as small as 2^-110: what
    was summed before it is not dropped."""
    s, at, scale = 300, 130, 1.0 / math.sqrt(d)
    q, k, v, g = (normal(280 + i, 2, s, d) for i in range(4))
    with_logit(q, k, at, logit, scale)
    v[:, at] = 0
    for name, r in everything(q, k, v, g, scale, causal).items():
        check_rows(f"late sink {logit} d{d} causal={causal} {name}", r, bar(logit + math.log(s)))
