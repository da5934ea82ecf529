"""The f16-pair kernels (csrc/fattn_pair.hip) where they can go wrong: the edges of their 32-row
tiles and 128 / 256-row workgroups, operands far from 1 and growing along the sequence (the
power-of-two scales), and values the split cannot carry (infinities, NaN), which go to the plain
fp32 rows. Everything against fp64 from plain torch on the same inputs."""
from __future__ import annotations

import math

import numpy as np
import pytest
import torch

import candle_fused_attn as cfa
import test_parity_gpu as parity

pytestmark = pytest.mark.gpu

# Normwise against fp64, as the parity tests' bar.
REL_TOL = 2e-6


def reference(q, k, v, scale, causal, g=None):
    """O (and dQ, dK, dV for the output gradient g) in fp64; q, k, v, g [n, s, d]."""
    q, k, v = (t.double().cpu() for t in (q, k, v))
    s = q.shape[1]
    x = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
    if causal:
        x = x.masked_fill(torch.ones(s, s, dtype=torch.bool).triu(1), -math.inf)
    p = torch.softmax(x, dim=-1)
    o = torch.matmul(p, v)
    if g is None:
        return [o]
    g = g.double().cpu()
    ds = p * (torch.matmul(g, v.transpose(1, 2).contiguous()) - (g * o).sum(-1, keepdim=True))
    return [o, torch.matmul(ds, k) * scale,
            torch.matmul(ds.transpose(1, 2).contiguous(), q) * scale,
            torch.matmul(p.transpose(1, 2).contiguous(), g)]


def rel(got, want):
    got = got.detach().double().cpu()
    return ((got - want).norm() / want.norm()).item()


def normal(seed, *shape):
    gen = torch.Generator(device="cuda:0").manual_seed(seed)
    return torch.randn(*shape, generator=gen, device="cuda:0")


def forward(q, k, v, scale, causal):
    with torch.no_grad():
        return cfa.fused_attention(q[None], k[None], v[None], scale, causal)[0]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("s", [1, 15, 17, 31, 32, 33, 64, 97, 127, 128, 129, 161, 257])
def test_forward_tile_edges(cuda, s, d, causal):
    q, k, v = (normal(7 * s + i, 3, s, d) for i in range(3))
    e = rel(forward(q, k, v, 0.125, causal), reference(q, k, v, 0.125, causal)[0])
    print(f"forward s{s} d{d} causal={causal}: {e:.2e}", flush=True)
    assert e <= REL_TOL


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("s", [33, 255, 256, 257])
def test_forward_wide_workgroups(cuda, s, d):
    """Two groups of 32 queries per wave (from 1024 workgroups of 256 queries on)."""
    n = 1024
    q, k, v = (normal(11 * s + i, n, s, d) for i in range(3))
    o = forward(q, k, v, 0.125, False)
    for i in (0, n // 2 + 1, n - 1):
        at = slice(i, i + 1)
        e = rel(o[at], reference(q[at], k[at], v[at], 0.125, False)[0])
        print(f"wide s{s} d{d} pair {i}: {e:.2e}", flush=True)
        assert e <= REL_TOL


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("n,s", [(1536, 32), (1024, 128), (1024, 129), (1024, 250), (511, 512),
                                 (512, 511), (512, 385), (512, 384), (205, 1153), (205, 1152)])
def test_forward_query_groups_rule(cuda, n, s, d):
    """One or two groups of 32 queries per wave, on either side of each condition of the choice (256
    queries per workgroup: how many of them, how many of their queries are padding)."""
    q, k, v = (normal(19 * s + i, n, s, d) for i in range(3))
    o = forward(q, k, v, 0.125, False)
    for i in (0, n // 2 + 1, n - 1):
        at = slice(i, i + 1)
        e = rel(o[at], reference(q[at], k[at], v[at], 0.125, False)[0])
        print(f"{n} x s{s} d{d} pair {i}: {e:.2e}", flush=True)
        assert e <= REL_TOL


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("qs,ks,vs,grow", [(1e-9, 1e9, 1e-12, 0), (1e6, 1e-7, 1e15, 0),
                                           (1.0, 1.0, 1e-3, 3), (1.0, 1.0, 1e3, -3)])
def test_forward_magnitudes(cuda, qs, ks, vs, grow, causal):
    """Operands far from 1, and V growing (or shrinking) by 2^grow from one 32-key tile to the
    next. Normwise over each 32-query block's rows, so that small rows count."""
    s, d = 200, 64
    q, k, v = (normal(40 + i, 2, s, d) * f for i, f in enumerate((qs, ks, vs)))
    v = v * torch.exp2(float(grow) * (torch.arange(s, device="cuda:0") // 32))[None, :, None]
    o = forward(q, k, v, 0.125, causal)
    want = reference(q, k, v, 0.125, causal)[0]
    for r in range(0, s, 32):
        e = rel(o[:, r:r + 32], want[:, r:r + 32])
        print(f"magnitudes rows {r}: {e:.2e}", flush=True)
        assert e <= REL_TOL


@pytest.mark.parametrize("d", [32, 64, 128])
def test_forward_non_finite(cuda, d):
    """An infinite key element makes scores +-inf (weight 0, or a NaN row), an infinite or NaN value
    reaches the rows that see it; every other row is untouched."""
    s = 150
    q, k, v = (normal(60 + i, 4, s, d) for i in range(3))
    k[0, 40, 3] = math.inf
    k[1, 130, 5] = -math.inf
    v[2, 100, 1] = math.nan
    v[3, 70, 2] = math.inf
    q[3, 9, 4] = math.nan
    for causal in (False, True):
        o = forward(q, k, v, 0.125, causal).double().cpu()
        want = reference(q, k, v, 0.125, causal)[0]
        if causal:
            # (0 weight times a non-finite value of a masked key is 0 here, NaN in the product.)
            for n, first in ((2, 100), (3, 70)):
                vv = v[n:n + 1].clone()
                vv[0, first] = 0
                want[n, :first] = reference(q[n:n + 1], k[n:n + 1], vv, 0.125, True)[0][0, :first]
        ok = torch.isfinite(want)
        assert torch.equal(torch.isfinite(o), ok), f"d{d} causal={causal}"
        assert torch.equal(torch.isnan(o), torch.isnan(want))
        e = ((o - want)[ok].norm() / want[ok].norm()).item()
        print(f"non-finite d{d} causal={causal}: {int(ok.sum())} of {ok.numel()} finite, {e:.2e}",
              flush=True)
        assert e <= REL_TOL


def gradients(q, k, v, g, scale, causal):
    """dQ, dK, dV [n, s, d] through the op."""
    q, k, v = (t[None].detach().requires_grad_() for t in (q, k, v))
    return [t[0] for t in torch.autograd.grad(cfa.fused_attention(q, k, v, scale, causal),
                                              (q, k, v), g[None])]


def check_gradients(got, want, what, tol=REL_TOL):
    for name, a, w in zip(("dq", "dk", "dv"), got, want):
        # (One key: P is 1 and dQ, dK are zero but for dP and D rounding apart.)
        e = rel(a, w) if w.shape[1] > 1 or name == "dv" else a.abs().max().item()
        print(f"{what} {name}: {e:.2e}", flush=True)
        assert e <= tol, (what, name)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("s", [1, 15, 17, 31, 32, 33, 64, 97, 127, 128, 129, 161, 257])
def test_backward_tile_edges(cuda, s, d, causal):
    q, k, v, g = (normal(13 * s + i, 3, s, d) for i in range(4))
    check_gradients(gradients(q, k, v, g, 0.125, causal),
                    reference(q, k, v, 0.125, causal, g)[1:], f"s{s} d{d} causal={causal}")


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("n", [32, 33])
def test_backward_serial_boundary(cuda, n, d):
    """Causal dV on either side of 64 key blocks, up to which it is summed in key order on the fp32
    matrix cores."""
    s = 256
    q, k, v, g = (normal(17 * n + i, n, s, d) for i in range(4))
    check_gradients(gradients(q, k, v, g, 0.125, True),
                    reference(q, k, v, 0.125, True, g)[1:], f"{n} pairs d{d}")


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("qs,ks,vs,gs,grow", [(1e-9, 1e9, 1e-12, 1e6, 0), (1e6, 1e-7, 1e9, 1e-9, 0),
                                              (1.0, 1.0, 1.0, 1.0, 3), (1.0, 1.0, 1.0, 1.0, -3)])
def test_backward_magnitudes(cuda, qs, ks, vs, gs, grow, causal):
    """Operands far from 1, and the output gradient growing (or shrinking) by 2^grow from one
    32-query tile to the next: dQ over each tile's rows, dK and dV normwise."""
    s, d = 200, 64
    q, k, v, g = (normal(80 + i, 2, s, d) * f for i, f in enumerate((qs, ks, vs, gs)))
    g = g * torch.exp2(float(grow) * (torch.arange(s, device="cuda:0") // 32))[None, :, None]
    got, want = gradients(q, k, v, g, 0.125, causal), reference(q, k, v, 0.125, causal, g)[1:]
    check_gradients(got, want, f"causal={causal}")
    for r in range(0, s, 32):
        check_gradients([got[0][:, r:r + 32]], [want[0][:, r:r + 32]], f"rows {r}")


@pytest.mark.parametrize("d", [32, 64, 128])
def test_backward_non_finite(cuda, d):
    """A NaN or infinite operand: non-finite gradients where the product has them, the values
    elsewhere, and the pairs that hold none untouched to the bit."""
    s = 150
    q, k, v, g = (normal(100 + i, 5, s, d) for i in range(4))
    clean = gradients(q, k, v, g, 0.125, False)
    k[0, 40, 3] = math.nan
    v[1, 100, 1] = math.inf
    q[2, 9, 4] = math.nan
    g[3, 149, 2] = -math.inf
    got, want = gradients(q, k, v, g, 0.125, False), reference(q, k, v, 0.125, False, g)[1:]
    for name, a, c, w in zip(("dq", "dk", "dv"), got, clean, want):
        a = a.double().cpu()
        assert torch.equal(a[4], c[4].double().cpu()), name
        ok = torch.isfinite(w)
        assert torch.equal(torch.isfinite(a), ok), name
        e = ((a - w)[ok].norm() / w[ok].norm()).item()
        print(f"non-finite d{d} {name}: {int(ok.sum())} of {ok.numel()} finite, {e:.2e}", flush=True)
        assert e <= REL_TOL, name


def test_backward_output_over_4gib(cuda):
    """One (b, h)'s rows of O spanning more than 4 GiB (the operands' rows do not)."""
    h, s, d = 8192, 1040, 128
    gen = torch.Generator(device="cuda:0").manual_seed(3)
    q, k, v, g = (torch.randn(h, s, d, generator=gen, device="cuda:0") for _ in range(4))
    got = gradients(q, k, v, g, 0.1, False)
    for i in (0, h - 1):
        at = slice(i, i + 1)
        check_gradients([t[at] for t in got], reference(q[at], k[at], v[at], 0.1, False, g[at])[1:],
                        f"head {i}")


@pytest.mark.parametrize("n", [3, 33])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_backward_zero_gradient(cuda, d, causal, n):
    """The output gradient zero for a whole pair, from a query on (a padded tail: whole key blocks
    see only zeros), and everywhere: gradients of exactly 0 where the products have nothing else.
    Causal, 3 and 33 pairs lie on either side of the serial dV rule."""
    s, tail = 256, 120
    q, k, v, g = (normal(120 + i, n, s, d) for i in range(4))
    g[0] = 0
    g[1, tail:] = 0
    got, want = gradients(q, k, v, g, 0.125, causal), reference(q, k, v, 0.125, causal, g)[1:]
    for a in got:
        assert torch.equal(a[0], torch.zeros_like(a[0]))
        if causal:
            assert torch.equal(a[1, tail:], torch.zeros_like(a[1, tail:]))
    check_gradients(got, want, f"zero gradient d{d} causal={causal}")
    for a in gradients(q, k, v, torch.zeros_like(g), 0.125, causal):
        assert torch.equal(a, torch.zeros_like(a))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_zero_operands(cuda, d, causal):
    """Each of q, k, v zero in turn: uniform weights, a zero output, and the gradients that are 0."""
    s = 130
    for which in range(3):
        q, k, v, g = (normal(140 + i, 2, s, d) for i in range(4))
        (q, k, v)[which].zero_()
        want = reference(q, k, v, 0.125, causal, g)
        got = [forward(q, k, v, 0.125, causal), *gradients(q, k, v, g, 0.125, causal)]
        for name, a, w in zip(("o", "dq", "dk", "dv"), got, want):
            if not w.any():
                assert torch.equal(a, torch.zeros_like(a)), (which, name)
                continue
            e = rel(a, w)
            print(f"operand {which} zero, d{d} causal={causal} {name}: {e:.2e}", flush=True)
            assert e <= REL_TOL, (which, name)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("f", [1e-28, 1e-30, 1e-32, 1e-35])
def test_tiny_magnitudes(cuda, f, causal):
    """Output gradients and values near the least normal float. Each result within the bar of its
    norm, or within one least subnormal (2^-149) per element where it is that small; dQ and dK of
    tiny values take the scale's bits off the bottom of that range."""
    s, d = 200, 64
    q, k, v, g = (normal(160 + i, 2, s, d) for i in range(4))

    def check(name, got, want):
        diff = (got.detach().double().cpu() - want).norm().item()
        floor = 2.0 ** -149 * math.sqrt(want.numel())
        print(f"{f:g} causal={causal} {name}: {diff / want.norm().item():.2e}", flush=True)
        assert diff <= REL_TOL * want.norm().item() + floor, name

    got, want = gradients(q, k, v, g * f, 0.125, causal), reference(q, k, v, 0.125, causal, g * f)
    for name, a, w in zip(("dq", "dk", "dv"), got, want[1:]):
        check(name, a, w)
    check("o", forward(q, k, v * f, 0.125, causal), reference(q, k, v * f, 0.125, causal)[0])


@pytest.mark.parametrize("s", [64, 150, 333])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_causal_non_finite_stays_in_its_rows(cuda, d, s):
    """Causal, a NaN or infinity in one row: the rows that do not see it are those of the same call
    with that row zero; queries and keys next to it in its tile among them."""
    at, scale = s // 2 + 3, 0.125
    x = [normal(180 + i, 1, s, d) for i in range(4)]
    before, after = slice(0, at), slice(at + 1, s)
    # (The infinite V reaches O, hence D, of every query from `at` on, but no P: dV stays whole.)
    unaffected = {"k": {"o": before, "dq": before}, "v": {"o": before, "dq": before, "dv": slice(0, s)},
                  "q": {"o": before, "dq": before, "dk": after, "dv": after},
                  "dO": {"dq": before, "dk": after, "dv": after}}
    for (name, rows), which, bad in zip(unaffected.items(), (1, 2, 0, 3),
                                        (math.nan, math.inf, math.inf, -math.inf)):
        y, z = [t.clone() for t in x], [t.clone() for t in x]
        y[which][0, at, 3] = bad
        z[which][0, at] = 0
        want = dict(zip(("o", "dq", "dk", "dv"), reference(*z[:3], scale, True, z[3])))
        got = dict(zip(("o", "dq", "dk", "dv"), [forward(*y[:3], scale, True),
                                                 *gradients(*y, scale, True)]))
        if name == "v":
            want["dv"] = reference(*x[:3], scale, True, x[3])[3]
        for out, r in rows.items():
            e = rel(got[out][:, r], want[out][:, r])
            print(f"{name} s{s} d{d} {out}: {e:.2e}", flush=True)
            assert e <= REL_TOL, (name, out)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("n,s", [(257, 1), (257, 31), (257, 32), (257, 33), (257, 63), (300, 64),
                                 (257, 65), (256, 32), (256, 64)])
def test_short_sequences_over_many_pairs(cuda, n, s, d, causal):
    """One, two or four waves per workgroup, on either side of s 32, s 64 and 256 (b, h): O and
    the gradients."""
    scale = 0.125
    q, k, v, g = (normal(23 * s + i, n, s, d) for i in range(4))
    o, got = forward(q, k, v, scale, causal), gradients(q, k, v, g, scale, causal)
    for i in (0, n // 2, n - 1):
        at = slice(i, i + 1)
        want = reference(q[at], k[at], v[at], scale, causal, g[at])
        e = rel(o[at], want[0])
        assert e <= REL_TOL
        check_gradients([t[at] for t in got], want[1:], f"{n} x s{s} d{d} causal={causal} o {e:.2e}")


@pytest.mark.parametrize("s", [32, 64])
def test_short_sequences_non_finite(cuda, s):
    """The fp32 rows in workgroups of one and two waves: one pair with an infinity, the others' bits
    those of a clean call."""
    n, d = 300, 64
    q, k, v, g = (normal(29 * s + i, n, s, d) for i in range(4))
    clean = [forward(q, k, v, 0.125, True), *gradients(q, k, v, g, 0.125, True)]
    v[5, s // 2, 3] = math.inf
    got = [forward(q, k, v, 0.125, True), *gradients(q, k, v, g, 0.125, True)]
    others = torch.arange(n, device="cuda:0") != 5
    for a, c in zip(got, clean):
        assert torch.equal(a[others], c[others])
    want = reference(q[5:6], k[5:6], v[5:6].nan_to_num(posinf=0.0), 0.125, True, g[5:6])
    assert rel(got[0][5:6, :s // 2], want[0][:, :s // 2]) <= REL_TOL
    assert rel(got[3][5:6], want[3]) <= REL_TOL


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("n,s", [(21, 257), (1, 640), (1, 2100)])
def test_backward_long_walks_of_small_grids(cuda, n, s, d):
    """Causal, few key blocks and walks past the serial rule's length: the same sum as in large grids,
    to the bit."""
    q, k, v, g = (normal(31 * s + i, n, s, d) for i in range(4))
    got = gradients(q, k, v, g, 0.125, True)
    check_gradients([t[:1] for t in got], reference(q[:1], k[:1], v[:1], 0.125, True, g[:1])[1:],
                    f"{n} x s{s} d{d}")
    more = -(-65 // ((s + 127) // 128))  # pairs of more than 64 key blocks
    many = gradients(*(t[:1].expand(more, s, d).contiguous() for t in (q, k, v, g)), 0.125, True)
    for a, w in zip(got, many):
        assert torch.equal(a[0], w[0])


@pytest.mark.parametrize("shape", [(2, 7, 3, 64), (2, 240, 6, 64), (1, 97, 2, 64), (1, 33, 2, 64),
                                   (2, 70, 3, 32), (1, 128, 2, 128), (2, 240, 3, 128)])
def test_closed_form_in_large_causal_grids(orc, cuda, shape):
    """The closed-form inputs of the reference's test in a batch of more than 64 key blocks, where the
    causal dV is not summed one query at a time: no component less accurate than 1.5 times the
    composed fp32 path against fp64."""
    b, s, h, d = shape
    x, w = orc.closed_form_inputs(b, s, h, d)
    want = parity.oracle_qkv(orc, x, w, h, d, True, np.float64)
    floor, cmax = parity.composed_floor(orc, x, w, h, d, True, want[0], want[2])
    copies = -(-65 // (b * h * ((s + 127) // 128)))
    qkv, wt = (torch.from_numpy(np.tile(t, (copies, 1, 1))).to(cuda) for t in (x, w))
    out, grad = (t[-b:] for t in parity.run("fused_qkv", qkv, wt, h, d, True))
    parity.check_errors(orc, out, grad, want[0], want[2], f"{copies} copies", floor, d=d)
    e = orc.max_abs(grad.cpu().numpy(), want[2])
    assert e <= max(parity.zero_band(d), 1.5 * cmax), f"max-abs {e:.3e}"


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("f", [1e-33, 1e-35])
@pytest.mark.parametrize("scale", [0.1, 0.003])
def test_tiny_gradients_under_any_scale(cuda, scale, f, causal):
    """As above with a scale that is no power of two: dQ and dK keep their bits where the factor that
    takes their sums back is subnormal."""
    s, d = 200, 64
    q, k, v, g = (normal(160 + i, 2, s, d) for i in range(4))
    got, want = gradients(q, k, v, g * f, scale, causal), reference(q, k, v, scale, causal, g * f)[1:]
    for name, a, w in zip(("dq", "dk", "dv"), got, want):
        diff = (a.double().cpu() - w).norm().item()
        print(f"{f:g} scale {scale} causal={causal} {name}: {diff / w.norm().item():.2e}", flush=True)
        assert diff <= REL_TOL * w.norm().item() + 2.0 ** -149 * math.sqrt(w.numel()), name


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("f", [1e-33, 1e33])
def test_tiny_against_huge(cuda, f, d, causal):
    """Queries and keys, values and output gradients of 1e-33 against 1e33: scores, and dP, of ordinary
    size."""
    s = 150
    q, k, v, g = (normal(300 + i, 2, s, d) * x for i, x in enumerate((f, 1 / f, f, 1 / f)))
    want = reference(q, k, v, 0.125, causal, g)
    got = [forward(q, k, v, 0.125, causal), *gradients(q, k, v, g, 0.125, causal)]
    for name, a, w in zip(("o", "dq", "dk", "dv"), got, want):
        e = rel(a, w)
        print(f"{f:g} d{d} causal={causal} {name}: {e:.2e}", flush=True)
        assert e <= REL_TOL, name
