"""What a plan's launches are issued as (the schedule is host code): which of
them share a kernel, and which must not."""
import pytest
import torch

from chatterbox_amdvulkan_amd import cbxops as C
from chatterbox_amdvulkan_amd import workloads as W
from chatterbox_amdvulkan_amd.cfm_estimator import CFMEstimator
from chatterbox_amdvulkan_amd.flow_encoder import FlowEncoderCall
from chatterbox_amdvulkan_amd.t3_decode import T3DecodeStep

from tests._steps import HostList, N_CU, kinds


def t3_step(n_past=255, layers=24):
    inp = W.t3_token_inputs(layers, 512)
    dev = {k: torch.from_numpy(v) for k, v in inp.items()}
    dev["token"] = dev["position"] = torch.zeros(1, dtype=torch.int32)
    return T3DecodeStep(dev, n_past)


def test_token_list():
    st = t3_step()
    steps = st.graph.steps(st.keep, N_CU)
    assert len(steps) == 4 and sum(len(s) for s in steps) == 121


def test_flow_and_estimator_lists():
    e = FlowEncoderCall(125, n_blocks=3, n_up_blocks=3, device=False)
    assert len(e.b.g.steps(e.keep, N_CU)) == 7
    e = CFMEstimator(500, n_mid=2, n_tr=2, device=False)
    plan, steps = e.b.g.plan(e.keep), e.b.g.steps(e.keep, N_CU)
    causal = [s for s in steps if plan[s[0]][0] == C.GL_CAUSAL_CONV1D]
    assert all(len(s) == 1 for s in causal) and len(causal) == 11 and len(steps) < 40


@pytest.mark.parametrize("ch,T", [(64, 12000), (128, 20000), (256, 4000)])
def test_layers_side_by_side(ch, T):
    """Three ResBlocks' independent layers: two launches of three layers."""
    l = HostList()
    x = l.x(T, ch)
    out = []
    for K in (3, 7, 11):
        y, _ = l.layer(x, ch, K, 1)
        y, _ = l.layer(y, ch, K, 3)
        out.append(y)
    steps = l.steps(out)
    assert [len(s) for s in steps] == [6, 6]
    assert kinds(l.g, out) == [[C.GL_CONV1D] * 6] * 2


def test_refuses_a_short_array():
    l = HostList()
    y = l.scale(l.x(4, 64), 2.0)
    assert l.steps([y]) == [[0]]
    T, N, _ = l.g._arrays([])
    n = C.ctypes.c_int32(0)
    assert C.load().cbx_graph_steps(T, 2, N, 1, None, 0, 64, None, 0, C.ctypes.byref(n)) == C.ERR_INVALID_ARG
    assert n.value == 1


# ---- buffers used again -----------------------------------------------------------

def step_of(l, keep, i):
    """The step whose launches make tensor i."""
    plan = l.g.plan(keep)
    for s, launches in enumerate(l.steps(keep)):
        if any(l.g.nodes[plan[k][1] + plan[k][2] - 1].dst == i for k in launches):
            return s
    raise AssertionError(i)


@pytest.mark.parametrize("bridge", ["x", "residual only"])
def test_layer_after_the_one_it_reads(bridge):
    """Layer 2 reads layer 1's result y1. Its first conv's output lies in the
    same arena, and an earlier tensor spans both: the class of bytes that the
    never-stored output is in holds y1 as well."""
    ch, T = 64, 12000
    n = ch * T
    l = HostList()
    arena = torch.empty(3 * n + 64)
    span = l.t(arena[:2 * n].view(2 * T, ch))
    dead = l.scale(span, 2.0)                                  # reads the arena before it is used again
    y1, _ = l.layer(l.x(T, ch), ch, 3, 1)
    if bridge == "x":
        l.place(y1, arena, 0)
        y2, h2 = l.layer(y1, ch, 3, 3)
    else:                                                      # x of its own, the residual is y1
        x2 = l.x(T, ch)
        y2, h2 = l.layer(x2, ch, 3, 3)
        l.place(y1, arena, 0)
        add = l.g.nodes[-1]
        add.src[0] = y1
    l.place(h2, arena, n)
    keep = [dead, y1, y2]
    assert step_of(l, keep, y1) < step_of(l, keep, y2)


def test_write_over_what_a_layer_reads():
    """A launch after the layer that writes over its input stays after it,
    also when an earlier step of its kind has room."""
    ch, T = 64, 12000
    n = ch * T
    l = HostList()
    arena = torch.empty(2 * n + 64)
    span = l.t(arena[:2 * n].view(2 * T, ch))
    early = l.scale(l.x(T, ch), 2.0)                           # an element-wise step ahead of the layer
    x = l.t(arena[:n].view(T, ch))
    y, h = l.layer(x, ch, 3, 1)
    l.place(h, arena, n)
    over = l.scale(l.x(T, ch), 3.0)                            # over x
    l.place(over, arena, 0)
    keep = [early, y, over]
    assert span >= 0 and step_of(l, keep, early) < step_of(l, keep, over)
    assert step_of(l, keep, y) < step_of(l, keep, over)


# ---- what an entry point refuses runs alone, where it is refused ----------------------

def bias_pair(l, T=64, D=512, heads=8):
    """add(x, bias) -> heads view -> add(., u), add(., v); the tensors by name."""
    t = {"x": l.x(T, D), "bias": l.x(D), "u": l.x(heads, D // heads), "v": l.x(heads, D // heads)}
    s = l.add(t["x"], t["bias"])
    w = l.node_view(l.at(s).view(T, heads, D // heads), s)
    t["yu"], t["yv"] = l.add(w, t["u"]), l.add(w, t["v"])
    return t


@pytest.mark.parametrize("out,over", [(None, None), ("yu", "yv"), ("yu", "v"), ("yv", "u"), ("yu", "u"), ("yv", "v"),
                                      ("yu", "bias"), ("yv", "x")])
def test_bias_pair_over_its_own_tensors(out, over):
    """cbx_bias_add_pair refuses an output over an input or the other output:
    such a launch joins no group (alone, it is refused)."""
    l = HostList()
    other = l.add(l.x(64, 512), l.x(512))
    l.scale(other, 2.0)
    t = bias_pair(l)
    if out:
        n = max(l.at(t[out]).numel(), l.at(t[over]).numel())
        buf = torch.empty(n + 64)
        # the graph's descriptors follow the tensors: views of x and the sum keep theirs
        for k in (out, over):
            l.place(t[k], buf, 0)
    keep = [other, t["yu"], t["yv"]]
    plan = l.g.plan(keep)
    pair = [i for i, p in enumerate(plan) if p[0] == C.GL_BIAS_ADD_PAIR]
    assert len(pair) == 1
    step, = [s for s in l.steps(keep) if pair[0] in s]
    assert (len(step) == 1) == bool(out)


def grouped(l, keep, dst):
    """Whether the launch making tensor dst shares its step."""
    plan = l.g.plan(keep)
    k, = [i for i, p in enumerate(plan) if l.g.nodes[p[1] + p[2] - 1].dst == dst]
    step, = [s for s in l.steps(keep) if k in s]
    return len(step) > 1


@pytest.mark.parametrize("form", ["add", "bias", "mask", "unary", "scale", "soft_max", "rows", "rows w", "concat"])
def test_descriptor_no_entry_point_takes(form):
    """A descriptor that every entry point refuses (reserved set) does not pass
    in a group's name."""
    l = HostList()
    T, D = 64, 256
    a = l.x(T, D)
    if form in ("add", "bias", "mask", "unary", "scale"):
        bad = l.x(*{"bias": (D,), "mask": (T, 1)}.get(form, (T, D)))
        first = l.scale(l.x(T, D), 2.0)
        y = (l.unary(bad, C.TANH) if form == "unary" else l.scale(bad, 2.0) if form == "scale"
             else l.mul(a, bad) if form == "mask" else l.add(a, bad))
    elif form == "soft_max":
        bad = l.x(8, T, T)
        first, y = l.soft_max(l.x(8, T, T)), l.soft_max(bad)
    elif form == "concat":
        bad = l.x(T, 80)
        first = l.concat(l.x(T, 80), bad, 0)
        y = l.concat(first, l.x(T, 80), 0)
    else:
        w = l.x(D)
        first = l.layer_norm(l.add(a, l.x(T, D)), l.x(D), l.x(D))
        bad = w if form == "rows w" else l.x(T, D)
        y = l.layer_norm(l.add(first, bad if form == "rows" else l.x(T, D)), w, l.x(D))
    keep = [y] if form == "concat" else [first, y]
    assert grouped(l, keep, y)
    l.g._descs[bad].reserved = 1
    assert not grouped(l, keep, y)


@pytest.mark.parametrize("what", ["type", "rows", "columns", "over a source"])
def test_concat_run_with_a_bad_intermediate(what):
    """cbx_concat would refuse the intermediate result: the concats run one by one."""
    l = HostList()
    T = 32
    srcs = [l.x(T, 80) for _ in range(3)]
    a = l.concat(srcs[0], srcs[1], 0)
    y = l.concat(a, srcs[2], 0)
    assert grouped(l, [y], y)
    d = l.g._descs[a]
    if what == "type":
        d.type = C.F16
    elif what == "rows":
        d.ne[1] = T + 1
    elif what == "columns":
        d.ne[0] = 176
    else:
        d.data = l.at(srcs[1]).data_ptr()
    assert not grouped(l, [y], y)


# ---- results left unstored ------------------------------------------------------------

def alias(l, i):
    """Tensor i's bytes under another descriptor, with no VIEW node."""
    return l.t(l.at(i))


@pytest.mark.parametrize("read", ["by a launch", "kept", "part of it", "after a write over it", "before it is made"])
def test_layer_whose_first_output_is_read_under_another_name(read):
    """conv1's output stays unstored only where no other descriptor of its
    bytes shows it: one that a later launch reads, or the caller keeps."""
    l = HostList()
    ch, T = 64, 12000
    x = l.x(T, ch)
    if read == "before it is made":
        buf = l.empty((T, ch))
        old = l.scale(l.t(buf), 2.0)
        y, h = l.layer(x, ch, 3, 1)
        l.g.rebind(h, buf)
        keep = [old, y]
    else:
        y, h = l.layer(x, ch, 3, 1)
        h2 = alias(l, h) if read != "part of it" else l.t(l.at(h).view(-1)[64:64 + 640].view(10, 64))
        keep = [y]
        if read == "kept":
            keep.append(h2)
        else:
            if read == "after a write over it":
                over = l.scale(l.x(T, ch), 3.0)
                l.g.rebind(over, l.at(h))
            keep.append(l.scale(h2, 2.0))
    fused = [s for s in kinds(l.g, keep) if s == [C.GL_CONV1D, C.GL_CONV1D]]
    assert len(fused) == (1 if read in ("after a write over it", "before it is made") else 0)


@pytest.mark.parametrize("read", [None, "by a launch", "kept"])
def test_concat_run_whose_middle_is_read_under_another_name(read):
    l = HostList()
    T = 32
    a = l.concat(l.x(T, 80), l.x(T, 80), 0)
    y = l.concat(a, l.x(T, 80), 0)
    keep = [y]
    if read == "kept":
        keep.append(alias(l, a))
    elif read:
        keep.append(l.unary(alias(l, a), C.TANH))
    assert any(s.count(C.GL_CONCAT) == 2 for s in kinds(l.g, keep)) == (read is None)


# ---- launch sizes ----------------------------------------------------------------------

class FarList(HostList):
    """Tensors that are descriptors only: addresses of their own and no memory."""

    @staticmethod
    def empty(shape, dtype=torch.float32):
        return torch.empty(shape, dtype=dtype, device="meta")

    def steps(self, keep, n_cu=N_CU):
        at, base = 1 << 44, {}
        for i, t in enumerate(self.g._torch):
            key = t.untyped_storage()._cdata
            if key not in base:
                base[key] = at
                at += -(-t.untyped_storage().nbytes() // 4096) * 4096 + 4096
            self.g._descs[i].data = base[key] + t.storage_offset() * t.element_size()
        return super().steps(keep, n_cu)


def test_group_of_more_work_items_than_a_grid_takes():
    """A grid holds under 2^32 work-items, and an element-wise group takes one
    a float4: of launches of 2^30 - 1 float4s, fewer than five share one."""
    l = FarList()
    keep = [l.scale(l.x((1 << 30) - 1, 4), 2.0) for _ in range(9)]
    steps = l.steps(keep)
    assert sum(len(s) for s in steps) == 9
    assert all(len(s) * (1 << 30) < 1 << 32 for s in steps)


@pytest.mark.parametrize("n,lg,shared", [(2, 19, 2), (2, 20, 0), (3, 20, 0), (4, 20, 4), (8, 20, 8), (8, 21, 0)])
def test_group_only_where_it_is_the_faster(n, lg, shared):
    """2^11 floats a launch and CU, twice that where four share it."""
    l = FarList()
    keep = [l.unary(l.add(l.x(1 << (lg - 10), 1024), l.x(1024)), C.GELU) for _ in range(n)]
    keep += [l.unary(l.add(l.x(1 << 14, 1024), l.x(1024)), C.GELU)]            # never
    steps = l.steps(keep)
    assert sum(len(s) for s in steps) == n + 1 and max(len(s) for s in steps) == max(shared, 1)
    assert [n] in steps


def test_group_of_whole_sums_and_concat_runs():
    """Four large sums of two whole tensors share a launch, two do not; a run
    of concats stays one launch whatever its size."""
    l = FarList()
    assert len(l.steps([l.add(l.x(4096, 1024), l.x(4096, 1024)) for _ in range(4)])) == 1
    l = FarList()
    assert len(l.steps([l.add(l.x(4096, 1024), l.x(4096, 1024)) for _ in range(2)])) == 2
    l = FarList()
    y = l.concat(l.concat(l.x(20000, 256), l.x(20000, 256), 0), l.x(20000, 256), 0)
    z = l.scale(l.x(8, 64), 2.0)
    assert sorted(len(s) for s in l.steps([y, z])) == [1, 2]
    l = FarList()
    y = l.concat(l.concat(l.x(200, 256), l.x(200, 256), 0), l.x(200, 256), 0)
    z = l.scale(l.x(8, 64), 2.0)
    assert [len(s) for s in l.steps([y, z])] == [3]


@pytest.mark.parametrize("rows", [1 << 26, 1 << 28])
def test_chain_of_more_rows_than_a_grid_takes(rows):
    """A chain takes at least 64 work-items a row, so under 2^26 rows; the
    launches alone take these."""
    l = FarList()
    j = l.add(l.x(rows, 4), l.add(l.x(rows, 4), l.x(4)))
    y = l.scale(j, 2.0)
    assert [p[0] for p in l.g.plan([j, y])] == [C.GL_BIAS_RESIDUAL, C.GL_SCALE]
    assert [len(s) for s in l.steps([j, y])] == [1, 1]


@pytest.mark.parametrize("T,D,n,chained", [(640, 1024, 2, True), (1000, 1024, 2, False), (1280, 512, 2, True),
                                           (2000, 512, 2, False), (2048, 256, 2, True), (2049, 80, 2, False),
                                           (1536, 1024, 4, True), (1537, 1024, 4, False), (6144, 80, 4, True),
                                           (6145, 80, 4, False)])
def test_chain_only_where_it_is_the_faster(T, D, n, chained):
    l = FarList()
    h, keep = l.x(T, D), []
    for _ in range(n):
        h = l.add(h, l.add(l.x(T, D), l.x(D)))
        keep.append(l.layer_norm(h, l.x(D), l.x(D)))
    assert [len(s) for s in l.steps(keep)] == ([n] if chained else [1] * n)


def test_large_launches_stay_in_the_lists_order():
    l = FarList()
    a = l.scale(l.x(8000, 512), 2.0)
    b = l.scale(a, 2.0)
    c = l.scale(l.x(8000, 512), 2.0)
    assert l.steps([b, c, a]) == [[0], [1], [2]]


@pytest.mark.parametrize("T,fused", [(1 << 20, True), (1 << 27, False)])
def test_layer_of_more_tiles_than_a_grid_takes(T, fused):
    """512 work-items a tile, three layers a launch: under 2^21 tiles each."""
    l = FarList()
    y, _ = l.layer(l.x(T, 256), 256, 3, 1)
    assert ([len(s) for s in l.steps([y])] == [2]) == fused


def test_unstored_intermediates_are_no_conflicts():
    """A result that no launch stores (the first layer's im2col) may lie over
    what two independent layers store: they share a launch all the same."""
    ch, T = 64, 12000
    l = HostList()
    ys = [l.layer(l.x(T, ch), ch, 3, 1)[0] for _ in range(2)]
    buf = torch.empty(2 * ch * T + 64)
    for k, y in enumerate(ys):
        l.place(y, buf, k * ch * T)
    assert [len(s) for s in l.steps(ys)] == [4]
    col = l.g.nodes[[i for i, n in enumerate(l.g.nodes) if n.op == C.GOP_IM2COL][0]].dst
    scratch = buf.view(torch.float16)[:3 * ch * T].view(l.at(col).shape)
    l.g.rebind(col, scratch)
    assert [len(s) for s in l.steps(ys)] == [4]
    # a read of both results together comes after them (and makes one class of
    # their bytes, so the layers keep their order too)
    over = l.scale(l.t(buf[:2 * ch * T].view(2 * T, ch)), 2.0)
    assert [len(s) for s in l.steps(ys + [over])] == [2, 2, 1]
