"""Node lists whose captured form issues several planned launches as one
kernel (element-wise groups, softmax groups, row chains: k_group.hip,
k_softmax.hip), against the same plan run launch by launch through
cbx_graph_launch on the same bytes: the kept tensors' bits are equal, replay
after replay, whatever the launches share."""
import ctypes

import pytest
import torch

from chatterbox_amdvulkan_amd import cbxops as C
from chatterbox_amdvulkan_amd.ggml_nodes import NodeList

pytestmark = pytest.mark.gpu


class Lists:
    """A node list over tensors this object can put back as they were."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)
        self.made = []
        self.b = NodeList(self.new)
        self.keep = []

    def new(self, shape, dtype):
        t = torch.full(shape, float("nan"), dtype=dtype, device="cuda")
        self.made.append(t)
        return t

    def x(self, *shape, std=1.0):
        t = torch.randn(shape, generator=self.gen, device="cuda") * std
        self.made.append(t)
        return self.b.t(t)

    def k(self, i):
        self.keep.append(i)
        return i

    def check(self, steps, replays=3):
        """steps: how many kernels the list is issued as on 256 CUs."""
        g, before = self.b.g, [t.clone() for t in self.made]
        T, N, _ = g._arrays(self.keep)
        plan = g.plan(self.keep)
        assert len(g.steps(self.keep)) == len(g.steps(self.keep, 256)) == steps
        for p in plan:
            rc = C.load().cbx_graph_launch(T, len(g._descs), N, len(g.nodes), ctypes.byref(C.GLaunch(*p)), C._stream())
            assert rc == C.OK, C.last_error()
        torch.cuda.synchronize()
        ref = [self.b.at(i).clone() for i in self.keep]
        ex = g.capture(self.keep)
        try:
            assert ex.n_launches == sum(1 for p in plan if p[0] != C.GL_VIEW)
            for rep in range(replays + 1):
                for t, s in zip(self.made, before):
                    t.copy_(s)
                if rep < replays:
                    ex.launch()
                else:
                    g.compute(self.keep)
                torch.cuda.synchronize()
                for i, r in zip(self.keep, ref):
                    got = self.b.at(i)
                    assert torch.equal(got.contiguous().view(torch.int32), r.contiguous().view(torch.int32)), \
                        f"pass {rep}, tensor {i} {tuple(got.shape)}: {int((got != r).sum())} values differ"
        finally:
            ex.close()


@pytest.mark.parametrize("T,D", [(1, 4), (3, 20), (125, 512), (500, 1024), (33, 2048)])
def test_elementwise(cbx, T, D):
    l = Lists(T * 10000 + D)
    b = l.b
    for act in (C.GELU, C.GELU_ERF, C.SILU, C.TANH, C.MISH, C.SQR):
        l.k(b.unary(b.add(l.x(T, D, std=4.0), l.x(D)), act))
        l.k(b.unary(l.x(T, D, std=4.0), act))
    l.k(b.add(l.x(T, D), l.x(T, D)))
    l.k(b.mul(l.x(T, D), l.x(T, D)))
    l.k(b.mul(l.x(T, D), l.x(T, 1)))
    l.k(b.add(l.x(T, D), l.x(T, 1)))
    l.k(b.add(l.x(T, D), l.x(D)))
    l.k(b.add(l.x(T, D), l.x(D)))
    l.k(b.scale(l.x(T, D), 0.37))
    l.k(b.leaky(l.x(T, D), 0.01))
    # a value per row on rows of T floats (any length): the (1, C) bias of a time-major tensor
    for _ in range(2):
        bias = l.x(D)
        l.k(b.add(l.x(D, T), b.node_view(b.at(bias).reshape(D, 1), bias)))
    # a chain of dependent element-wise launches behind them
    y = l.k(b.scale(l.x(T, D), 2.0))
    y = l.k(b.add(y, l.x(T, D)))
    l.k(b.unary(y, C.TANH))
    l.check(3)


@pytest.mark.parametrize("parts,kept,steps", [((4, 4), (), 1), ((8, 80, 4), (), 1), ((80, 80, 80, 80), (), 1),
                                              ((256, 4, 12, 8, 16), (), 1), ((4,) * 9, (), 2),
                                              ((80, 80, 80, 80), (1,), 2), ((80, 3, 5, 80), (), 3)])
def test_concats(cbx, parts, kept, steps):
    """Runs of concats along dim 0: only the last result is stored unless a
    caller keeps one between; odd widths run as they are."""
    l = Lists(sum(parts))
    b, T = l.b, 37
    y = l.x(T, parts[0])
    for n, w in enumerate(parts[1:]):
        y = b.concat(y, l.x(T, w), 0)
        if n in kept:
            l.k(y)
    l.k(y)
    l.k(b.scale(l.x(T, 64), 3.0))
    l.check(steps)


@pytest.mark.parametrize("heads,q,kv,steps", [(8, 125, 125, 3), (8, 250, 250, 3), (16, 1, 257, 3), (8, 300, 300, 3),
                                              (3, 7, 1100, 10), (8, 500, 77, 3)])
def test_softmaxes(cbx, heads, q, kv, steps):
    l = Lists(heads * q + kv)
    b = l.b
    for n in range(5):
        l.k(b.soft_max(b.scale(l.x(heads, q, kv, std=5.0), 0.125 * (n + 1))))
    for _ in range(2):
        l.k(b.soft_max(b.scale(b.add(l.x(heads, q, kv, std=5.0), l.x(heads, q, kv, std=5.0)), 0.125)))
    m = b.node_new(C.GOP_DIAG_MASK_INF, (heads, q, kv), (l.x(heads, q, kv),), iparam=max(0, kv - q))
    l.k(b.soft_max(m))
    # another length with the same rows, and one that reads a softmax
    l.k(b.soft_max(b.scale(l.x(heads, q, kv + 4), 0.5)))
    l.k(b.soft_max(b.scale(l.keep[0], 2.0)))
    l.check(steps)


def ln(l, x, eps=1e-5):
    D = l.b.shape(x)[-1]
    return l.b.layer_norm(x, l.x(D), l.x(D), eps)


# one wave a row, several, one row to several rounds of rows, more links than
# a chain holds; rows longer than a chain takes, and more floats than one is
# the faster for
@pytest.mark.parametrize("T,D,n,steps", [(1, 1024, 30, 4), (3, 4, 3, 3), (500, 256, 4, 3), (125, 512, 5, 3), (250, 260, 2, 3),
                                         (2100, 512, 3, 5), (2100, 1024, 2, 13), (7, 768, 4, 3), (20, 1028, 2, 11)])
def test_row_chain(cbx, T, D, n, steps):
    l = Lists(T + D + n)
    b = l.b
    mask = b.t((torch.rand((T, 1), generator=l.gen, device="cuda") > 0.2).float())
    h = l.k(b.mul(b.mish(ln(l, l.x(T, D))), mask))
    tm = b.add(l.x(D), l.x(D))
    h = b.add(h, b.node_view(b.at(tm).reshape(1, D), tm))
    l.k(b.scale(ln(l, h), 1.7))
    for i in range(n):
        h = b.add(h, b.add(l.x(T, D), l.x(D)))        # residual join, its sum kept in some links
        l.k(ln(l, h, 1e-12))
        if i % 3 == 0:
            l.k(h)
        h2 = b.add(l.x(T, D), h)
        l.k(ln(l, h2))
        l.k(b.mul(h2, mask))
        l.k(b.unary(b.add(l.x(T, 2 * D), l.x(2 * D)), C.GELU))
        h = h2
    l.k(b.add(h, b.add(l.x(T, D), l.x(D))))
    l.check(steps)


def test_shared_buffers(cbx):
    """Results that take over the bytes of earlier tensors (in place, or a
    buffer used again, whole or in part): the order of the list holds, while
    the launches between them that touch none of it share one kernel."""
    T, D = 64, 256
    l = Lists(11)
    b, g = l.b, l.b.g
    buf = torch.zeros(4 * T * D, device="cuda")
    l.made.append(buf)

    def at(off, rows=T, cols=D):
        return b.t(buf[off:off + rows * cols].view(rows, cols))

    def add(dst, x, y):
        g.node(C.GOP_ADD, dst, (x, y))
        return dst

    def aside():
        l.k(b.scale(l.x(T, D), 1.5))

    n = T * D
    a = add(at(0), l.x(T, D), l.x(T, D))
    c = l.k(b.scale(a, 2.0))
    aside()
    d = add(at(0), l.x(T, D), l.x(T, D))              # over a, read above
    l.k(b.mul(d, c))
    aside()
    e = add(at(n // 2), l.x(T, D), l.x(D))            # half over d
    l.k(ln(l, e))
    aside()
    f = add(e, e, l.x(T, D))                          # in place
    h = l.k(ln(l, f))
    aside()
    s = add(at(n), f, h)
    l.k(ln(l, s))
    aside()
    s2 = add(at(n), s, l.x(T, D))                     # the sum in place, its norm next
    l.k(ln(l, s2))
    l.k(b.soft_max(b.scale(s2, 0.5)))
    aside()
    add(at(n), l.x(T, D), l.x(T, D))                  # over s2 after its readers
    l.k(at(0))
    l.k(at(n))
    l.k(at(n // 2))
    l.check(10)


def test_misaligned_rows_run_alone(cbx):
    T, D = 50, 256
    l = Lists(12)
    b = l.b
    odd = torch.randn(T * D + 1, device="cuda")
    l.made.append(odd)
    x = b.t(odd[1:].view(T, D))
    for _ in range(2):
        l.k(b.unary(b.add(l.x(T, D), l.x(D)), C.SILU))
        l.k(b.add(x, l.x(T, D)))
        l.k(b.scale(x, 2.0))
    l.k(b.soft_max(b.scale(x, 0.3)))
    l.k(b.soft_max(b.scale(l.x(T, D), 0.3)))
    l.check(6)


def test_update_moves_between_steps(cbx):
    """An update that makes a launch depend on another regroups; the results
    are those of the new list."""
    T, D = 32, 128
    l = Lists(13)
    b, g = l.b, l.b.g
    x, y = l.x(T, D), l.x(T, D)
    p = l.k(b.scale(x, 2.0))
    q = l.k(b.scale(y, 3.0))
    ex = g.capture(l.keep)
    ex.launch()
    torch.cuda.synchronize()
    assert torch.equal(b.at(q), b.at(y) * 3.0)
    n = g.nodes[-1]
    for src in (p, y, p):
        n.src[0] = src
        b.at(q).fill_(float("nan"))
        ex.update(keep=l.keep)
        for _ in range(2):
            ex.launch()
        torch.cuda.synchronize()
        assert torch.equal(b.at(p), b.at(x) * 2.0) and torch.equal(b.at(q), b.at(src) * 3.0)
    ex.close()
