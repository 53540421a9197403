"""The one-launch ResBlock layers (k_resblock.hip) that a captured node list
runs in place of two convs each, against the same arithmetic in float64:
operands rounded to f16 where the convs round them, everything else exact.

Bounds.  An operand whose f32 value lies within an f32 error of a rounding
boundary may land one f16 ulp off (2^-10 of it), so an output differs by at
most 2^-10 sum |w s| of each conv (the first one's through the second's
weights; |snake'| <= 1 + alpha * alpha_inv = 2 for the alphas used) and the
f32 sums' 2^-18 of the same; the few such operands leave the 2-norm of the
difference under 1e-4 of the result's."""
import math

import pytest
import torch

from chatterbox_amdvulkan_amd import cbxops as C
from chatterbox_amdvulkan_amd.ggml_nodes import NodeList

pytestmark = pytest.mark.gpu


def rnd(g, *shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda") * std


def params(g, ch, K, alpha=None):
    p = {}
    for i in ("1", "2"):
        a = torch.rand((ch,), generator=g, device="cuda") + 0.5
        ai = 1.0 / (a + 1e-9)
        if alpha is not None:
            a[::7], ai[::7] = alpha, 2.0 ** -14
        p["a" + i], p["ai" + i] = a, ai
        p["w" + i] = rnd(g, ch, ch, K, std=1.0 / math.sqrt(ch * K))
        p["b" + i] = rnd(g, ch, std=0.1)
    return p


def conv(x, w, d):
    co, ci, K = w.shape
    T, pad = x.shape[0], (K - 1) // 2 * d
    xp = torch.zeros((T + 2 * pad, ci), dtype=torch.float64, device=x.device)
    xp[pad:pad + T] = x
    y = torch.zeros((T, co), dtype=torch.float64, device=x.device)
    for j in range(K):
        y += xp[j * d:j * d + T] @ w[:, :, j].t().contiguous()
    return y


def f16(x):
    return x.half().double()


def snake16(x, a, ai):
    """f16 of x + sin(x a)^2 a_inv, the product x a in f32 as the kernel takes it."""
    xf = x.float()
    return f16((xf.double() + torch.sin((xf * a).double()) ** 2 * ai.double()).float())


def layer(x, p, d):
    """(y, bound) of one layer."""
    w1, w2 = f16(p["w1"]), f16(p["w2"])
    s1 = snake16(x, p["a1"], p["ai1"])
    h = conv(s1, w1, d) + p["b1"].double()
    s2 = snake16(h, p["a2"], p["ai2"])
    y = x + conv(s2, w2, 1) + p["b2"].double()
    eps = 2.0 ** -10 + 2.0 ** -18
    dh = eps * conv(s1.abs(), w1.abs(), d)
    return y, conv(eps * s2.abs() + 2 * dh, w2.abs(), 1) + 2.0 ** -20 * y.abs()


def new(shape, dtype):
    return torch.full(shape, float("nan"), dtype=dtype, device="cuda")


def add_layer(b, x, p, d, convs):
    cw = [C.Conv1dWeights(p["w1"]), C.Conv1dWeights(p["w2"])]
    convs += cw
    return b.sublayer(x, {n: b.t(t) for n, t in p.items()}, d, *cw)


def replay(b, keep, convs, steps, n=2):
    """steps: how many kernels the list is issued as on 256 CUs."""
    assert len(b.g.steps(keep)) == steps
    ex = b.g.capture(keep)
    try:
        for _ in range(n):
            for i in keep:
                b.at(i).fill_(float("nan"))
            ex.launch()
            torch.cuda.synchronize()
        return [b.at(i).double() for i in keep]
    finally:
        ex.close()
        for c in convs:
            c.close()


def check(got, ref, bound, what):
    d = (got - ref).abs()
    assert torch.isfinite(got).all(), what
    assert not (d > bound).any(), f"{what}: {int((d > bound).sum())} off, worst {float((d / bound).max()):.3g} of the bound"
    rel = float((got - ref).norm() / ref.norm())
    assert rel < 1e-4, f"{what}: rel {rel:.3g}"


# frames: whole tiles, one frame over, one short, and where the launch starts
# to be taken (32 tiles, 86 for K 11, 86 and 171 at 256 channels)
@pytest.mark.parametrize("ch,K,d,T", [
    (64, 3, 1, 126 * 32), (64, 3, 5, 126 * 33 + 1), (64, 7, 3, 122 * 40 - 1), (64, 11, 5, 118 * 86 + 7),
    (128, 3, 3, 62 * 32), (128, 7, 5, 58 * 33 + 1), (128, 11, 1, 54 * 87 - 1),
    (256, 3, 1, 30 * 33 + 1), (256, 7, 5, 26 * 86), (256, 11, 3, 22 * 171 - 1), (64, 1, 1, 128 * 32 + 3)])
def test_layer(cbx, ch, K, d, T):
    g = torch.Generator(device="cuda")
    g.manual_seed(ch * 1000 + K * 10 + d)
    p, x, convs = params(g, ch, K), rnd(g, T, ch), []
    b = NodeList(new)
    y = add_layer(b, b.t(x), p, d, convs)
    got, = replay(b, [y], convs, steps=1)
    ref, bound = layer(x.double(), p, d)
    check(got, ref, bound, f"{ch} x {T} K {K} d {d}")


@pytest.mark.parametrize("ch,T", [(64, 126 * 100 + 5), (128, 62 * 100 + 5), (256, 30 * 180 + 5)])
def test_three_blocks_and_their_sum(cbx, ch, T):
    """A stage's ResBlocks (K 3, 7, 11) side by side, the sum and its scale
    in the last layers' stores; the first block's output kept as well."""
    g = torch.Generator(device="cuda")
    g.manual_seed(ch)
    x, convs, total = rnd(g, T, ch), [], None
    b = NodeList(new)
    xi = b.t(x)
    ref = bound = None
    for K in (3, 7, 11):
        r, rr, rb = xi, x.double(), 0.0
        for d in (1, 3):
            p = params(g, ch, K)
            r = add_layer(b, r, p, d, convs)
            rr, nb = layer(rr.float().double(), p, d)
            # the incoming difference through both convs of this layer
            rb = nb if d == 1 else rb + nb + 4 * conv(conv(rb, p["w1"].double().abs(), d), p["w2"].double().abs(), 1)
        if total is None:
            first, first_ref, first_bound = r, rr, rb
        total = r if total is None else b.add(total, r)
        ref = rr if ref is None else ref + rr
        bound = rb if bound is None else bound + rb
    y = b.scale(total, 1.0 / 3.0)
    # the first layers share a launch; the sum runs through the second ones
    outs = replay(b, [first, y], convs, steps=4)
    for got, exp, bd in zip(outs, (first_ref, ref / 3.0), (first_bound, bound)):
        assert torch.isfinite(got).all() and not ((got - exp).abs() > bd).any()
        # an f16 operand flipped in layer one flips more in layer two: a few 1e-4
        assert float((got - exp).norm() / exp.norm()) < 1e-3


def test_large_arguments(cbx):
    """Arguments of sin at and past 2^16 take the library sinf, in the input
    window and in the intermediate (there |x a| is in f32 what the sums give,
    so the sine is free: its weight is 2^-14)."""
    ch, K, d, T = 128, 3, 1, 62 * 33
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    p, x, convs = params(g, ch, K, alpha=2.0 ** 18), rnd(g, T, ch), []
    b = NodeList(new)
    y = add_layer(b, b.t(x), p, d, convs)
    got, = replay(b, [y], convs, steps=1)
    ref, bound = layer(x.double(), p, d)
    free = torch.zeros(T, ch, dtype=torch.float64, device="cuda")
    free[:, ::7] = 2.0 ** -14
    bound = bound + conv(free, f16(p["w2"]).abs(), 1)
    assert torch.isfinite(got).all() and not ((got - ref).abs() > bound).any()


def test_infinite_input_stays_in_its_reach(cbx):
    ch, K, d, T, t = 64, 7, 3, 122 * 40, 2440
    g = torch.Generator(device="cuda")
    g.manual_seed(6)
    p, x, convs = params(g, ch, K), rnd(g, T, ch), []
    x[t, 9] = float("inf")
    b = NodeList(new)
    y = add_layer(b, b.t(x), p, d, convs)
    got, = replay(b, [y], convs, steps=1)
    bad = ~torch.isfinite(got).all(1)
    lo, hi = t - 3 * d - 3, t + 3 * d + 3
    assert not bad[:lo].any() and not bad[hi + 1:].any() and bool(bad[t])


@pytest.mark.parametrize("how", ["kept", "misaligned", "in place"])
def test_layers_the_launch_leaves_alone(cbx, how):
    """A kept intermediate, rows off 16 bytes, and an output over the residual
    run as two convs, with the same result."""
    ch, K, d, T = 64, 3, 1, 126 * 40
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    p, x0, convs = params(g, ch, K), rnd(g, T, ch), []
    x = x0.clone()
    if how == "misaligned":
        x = torch.empty(T * ch + 1, device="cuda")[1:].view(T, ch)
        x.copy_(x0)
    b = NodeList(new)
    xi = b.t(x)
    y = add_layer(b, xi, p, d, convs)
    keep = [y]
    if how == "kept":
        h = b.g.nodes[[i for i, n in enumerate(b.g.nodes) if n.op == C.GOP_UNARY and n.iparam == C.SIN][1] - 1].src[0]
        keep = [h, y]
    if how == "in place":
        dst = b.t(x)
        b.g.nodes[-1].dst = dst
        assert len(b.g.steps([dst])) == 2
        ex = b.g.capture([dst])
        ex.launch()
        torch.cuda.synchronize()
        got = b.at(dst).double()
        ex.close()
        for c in convs:
            c.close()
    else:
        got = replay(b, keep, convs, steps=2)[-1]
    ref, bound = layer(x0.double(), p, d)
    check(got, ref, bound, how)


@pytest.mark.parametrize("ch,T", [(64, 126 * 60 + 5), (128, 62 * 60 + 5)])
def test_layers_over_buffers_used_again(cbx, ch, T):
    """Layer 2 reads layer 1's result, beside which its own first conv's output
    lies in one arena that an earlier tensor spans; a later launch writes over
    that result."""
    g = torch.Generator(device="cuda")
    g.manual_seed(ch + 1)
    p1, p2, x, convs = params(g, ch, 3), params(g, ch, 3), rnd(g, T, ch), []
    arena = torch.empty(2 * T * ch, device="cuda")
    b = NodeList(new)
    span = b.t(arena.view(2 * T, ch))
    dead = b.scale(span, 2.0)
    y1 = add_layer(b, b.t(x), p1, 1, convs)
    b.g.rebind(y1, arena[:T * ch].view(T, ch))
    n = len(b.g.nodes)
    y2 = add_layer(b, y1, p2, 3, convs)
    sin = [i for i in range(n, len(b.g.nodes)) if b.g.nodes[i].op == C.GOP_UNARY and b.g.nodes[i].iparam == C.SIN][1]
    b.g.rebind(b.g.nodes[sin - 1].src[0], arena[T * ch:].view(T, ch))
    over = b.scale(b.t(x), 3.0)
    b.g.rebind(over, arena[:T * ch].view(T, ch))
    assert [len(s) for s in b.g.steps([dead, y2, over])] == [1, 2, 2, 1]
    ex = b.g.capture([dead, y2, over])
    for _ in range(2):
        arena.fill_(1.0)
        b.at(y2).fill_(float("nan"))
        ex.launch()
        torch.cuda.synchronize()
        r1, bound1 = layer(x.double(), p1, 1)
        r2, bound2 = layer(r1.float().double(), p2, 3)
        w1 = p2["w1"].double().abs()
        bound = bound1 + bound2 + 4 * conv(conv(bound1, w1, 3), p2["w2"].double().abs(), 1)
        got = b.at(y2).double()
        assert torch.isfinite(got).all() and not ((got - r2).abs() > bound).any()
        assert torch.equal(b.at(over), x * 3.0) and bool((b.at(dead) == 2.0).all())
    ex.close()
    for c in convs:
        c.close()
