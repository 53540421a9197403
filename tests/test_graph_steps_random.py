"""Random node lists over memory used again, carried out symbolically in the
list's order and as the steps they are issued as: every kept tensor holds the
same values, and no step reads what another launch of it writes.

Memory is a map from 64-byte units to values; a launch's value is its number
and everything it reads.  What a launch loads and stores is worked out here
from the nodes alone."""
import random

import pytest
import torch

from chatterbox_amdvulkan_amd import cbxops as C

from tests._steps import HostList

N_CU = 8            # few CUs: small tensors reach every form's limits
UNIT = 64


class ArenaList(HostList):
    def __init__(self, rng, share):
        self.rng, self.share = rng, share
        self.mem = torch.empty(40 * 64 * 64 * 4 + UNIT, dtype=torch.uint8)
        self.off0 = -self.mem.data_ptr() % UNIT
        super().__init__()

    def empty(self, shape, dtype=torch.float32):
        n = 1
        for s in shape:
            n *= s
        size = n * torch.empty(0, dtype=dtype).element_size()
        if self.rng.random() < self.share and size <= 8 * 64 * 64 * 4:
            # mostly at whole tensors' places, now and then half over two
            at = self.rng.randrange(0, 24) * 64 * 64 * 2 * self.rng.choice([1, 2])
            at = self.off0 + at % (32 * 64 * 64 * 4)
            return self.mem[at:at + size].view(dtype).view(shape)
        raw = torch.empty(size + 2 * UNIT, dtype=torch.uint8)
        at = -raw.data_ptr() % UNIT
        return raw[at:at + size].view(dtype).view(shape)


    def params(self, ch, K):
        share, self.share = self.share, 0.0     # (a layer's weights are prepared copies: not memory of the list)
        p = super().params(ch, K)
        self.share = share
        return p


def build(rng):
    l = ArenaList(rng, rng.choice([0.0, 0.2, 0.6, 0.9]))
    T, D = rng.choice([(64, 64), (32, 64), (16, 128), (64, 128)])
    pool = [l.x(T, D) for _ in range(3)]
    keep = []

    def pick():
        return rng.choice(pool[-4:] if rng.random() < 0.6 else pool)

    for _ in range(rng.randint(4, 24)):
        op = rng.choice(["add", "add", "bias", "act", "scale", "mul", "mask", "ln", "join", "joinb", "softmax", "concat",
                         "alias", "inplace", "pair", "biasres", "layer", "copy"])
        if op == "add":
            y = l.add(pick(), pick())
        elif op == "bias":
            y = l.add(pick(), l.x(D))
        elif op == "act":
            y = l.unary(l.add(pick(), l.x(D)), rng.choice([C.GELU, C.TANH, C.SILU]))
        elif op == "scale":
            y = l.scale(pick(), 0.5)
        elif op == "mul":
            y = l.mul(pick(), pick())
        elif op == "mask":
            y = l.mul(pick(), l.x(T, 1))
        elif op == "ln":
            y = l.layer_norm(pick(), l.x(D), l.x(D))
            if rng.random() < 0.5:
                y = l.scale(y, 1.5) if rng.random() < 0.5 else l.mul(l.mish(y), l.x(T, 1))
        elif op in ("join", "joinb"):
            h = l.add(pick(), l.x(D)) if op == "joinb" else pick()
            h = l.add(h, pick())
            y = l.layer_norm(h, l.x(D), l.x(D))
            pool.append(h)
        elif op == "softmax":
            y = l.soft_max(l.scale(l.add(pick(), pick()) if rng.random() < 0.3 else pick(), 0.25))
        elif op == "concat":
            y = pick()
            for _ in range(rng.randint(1, 3)):
                y = l.concat(y, pick(), 0)
                if rng.random() < 0.2:
                    keep.append(y)
            keep.append(y)
            continue
        elif op == "alias":
            y = l.t(l.at(pick()))
        elif op == "inplace":
            x = pick()
            y = l.scale(x, 3.0) if rng.random() < 0.5 else l.add(x, pick())
            l.g.rebind(y, l.at(x))
        elif op == "pair":
            x, b = pick(), l.x(D)
            s = l.add(x, b)
            w = l.node_view(l.at(s).view(T, 4, D // 4), s)
            u, v = l.x(4, D // 4), l.x(4, D // 4)
            keep += [l.add(w, u), l.add(w, v)]
            continue
        elif op == "biasres":
            y = l.add(pick(), l.add(pick(), l.x(D)))
        elif op == "layer":
            if D != 64:
                continue
            y, h = l.layer(pick(), 64, 3, rng.choice([1, 3]))
            if rng.random() < 0.3:
                pool.append(l.t(l.at(h).view(T, D)))
        else:
            y = l.node_new(C.GOP_CPY, (T, D), (pick(),))
        pool.append(y)
        if rng.random() < 0.4:
            keep.append(y)
    made = {n.dst for n in l.g.nodes}
    keep = [k for k in dict.fromkeys(keep) if k in made or rng.random() < 0.5]
    last = l.g.nodes[-1].dst if l.g.nodes else None
    return l, keep + ([last] if last is not None and last not in keep else [])


class Machine:
    def __init__(self, l, keep):
        self.l, self.keep, self.nodes, self.plan = l, keep, l.g.nodes, l.g.plan(keep)
        uses = {}
        for n in self.nodes:
            for s in n.src:
                uses[s] = uses.get(s, 0) + 1
        self.rd, self.wr, self.out = [], [], []
        for kind, f, cnt, flags in self.plan:
            nd, rd, wr = self.nodes[f:f + cnt], [], []
            for k, n in enumerate(nd):
                rd += [s for s in n.src if s >= 0 and s not in [m.dst for m in nd[:k]] and s not in rd]
                inside = sum(list(m.src).count(n.dst) for m in nd[k + 1:])
                if n.op != C.GOP_VIEW and not (inside and inside == uses[n.dst] and n.dst not in keep and k + 1 < cnt):
                    wr.append(n.dst)
            if kind == C.GL_VIEW:
                rd, wr = [], []
            if kind == C.GL_ADD_LAYER_NORM:
                assert (len(wr) == 1) == bool(flags & 1)
            self.rd.append(rd)
            self.wr.append(wr)
            self.out.append(nd[-1].dst)

    def units(self, i):
        d = self.l.g._descs[i]
        n = d.ne[0] * d.ne[1] * d.ne[2] * d.ne[3] * self.l.at(i).element_size()
        return range(d.data // UNIT, (d.data + n - 1) // UNIT + 1)

    def values(self, mem, i, own):
        if i in own:
            return own[i]
        return tuple(mem.get(u, u) for u in self.units(i))

    def result(self, k, mem, own):
        """Launch k's stored tensors -> the values of their units."""
        key = hash((k,) + tuple(self.values(mem, i, own) for i in self.rd[k]))
        return {i: tuple(hash((key, i, n)) for n in range(len(self.units(i)))) for i in self.wr[k]}

    def store(self, mem, res):
        for i, v in res.items():
            mem.update(zip(self.units(i), v))

    def in_order(self):
        mem = {}
        for k in range(len(self.plan)):
            self.store(mem, self.result(k, mem, {}))
        return [self.values(mem, i, {}) for i in self.keep]

    def meets(self, a, b):
        u, v = self.units(a), self.units(b)
        return u.start < v.stop and v.start < u.stop

    def fused(self, step):
        """The step's entries: launches, or runs of which only the last result is stored."""
        kind, out = [self.plan[k][0] for k in step], []
        for p, k in enumerate(step):
            conv2 = kind[p] == C.GL_CONV1D and len(step) > 1 and p % 2 == 1
            run = (kind[p] == C.GL_CONCAT and p > 0 and step[p - 1] == k - 1 and kind[p - 1] == C.GL_CONCAT
                   and self.nodes[self.plan[k][1]].src[0] == self.out[k - 1])
            if conv2 or run:
                out[-1].append(k)
            else:
                out.append([k])
        return out

    def as_steps(self):
        mem = {}
        steps = self.l.g.steps(self.keep, N_CU)
        assert sorted(k for s in steps for k in s) == [k for k, p in enumerate(self.plan) if p[0] != C.GL_VIEW]
        for step in steps:
            entries = self.fused(step)
            chain = len(step) > 1 and any(set(self.rd[b]) & set(self.wr[a]) or
                                          any(self.meets(x, y) for x in self.rd[b] for y in self.wr[a])
                                          for n, b in enumerate(step) for a in step[:n]) and len(entries) == len(step)
            if chain:
                self.check_chain(step)
                for k in step:
                    self.store(mem, self.result(k, mem, {}))
                continue
            done = []
            for e in entries:
                own, reads = {}, []
                for k in e:
                    reads += [i for i in self.rd[k] if i not in own]
                    res = self.result(k, mem, own)
                    if k != e[-1]:
                        own.update(res)
                done.append((e, reads, res))
            for e, reads, res in done:
                for e2, reads2, res2 in done:
                    if e2 is not e:
                        assert not any(self.meets(w, x) for w in res for x in list(reads2) + list(res2)), (step, e, e2)
                if len(step) > 1:      # in place at most, element for element
                    for w in res:
                        for x in reads:
                            assert not self.meets(w, x) or self.units(w) == self.units(x), (step, e)
            for _, _, res in done:
                self.store(mem, res)
        return [self.values(mem, i, {}) for i in self.keep], steps

    def check_chain(self, step):
        """A link reads earlier links' stores only as the last one's, whole,
        and stores over nothing that the chain reads or stores."""
        for n, k in enumerate(step):
            last = list(self.wr[step[n - 1]]) if n else []
            kind, f = self.plan[step[n - 1]][:2]
            if n and kind in (C.GL_LAYER_NORM, C.GL_LAYER_NORM_MASK, C.GL_SCALE, C.GL_BINARY):
                last.append(self.nodes[f].src[0])      # a link without a sum of its own still holds its operand
            fwd = [self.units(i) for i in last]
            for x in self.rd[k]:
                if any(self.meets(x, w) for a in step[:n] for w in self.wr[a]):
                    assert self.units(x) in fwd, (step, k, x)
            for w in self.wr[k]:
                for a in step[:n + 1]:
                    assert not any(self.meets(w, x) for x in self.rd[a]), (step, k, w)
                    assert a == k or not any(self.meets(w, x) for x in self.wr[a]), (step, k, w)


@pytest.mark.parametrize("block", range(8))
def test_steps_give_the_lists_values(block):
    shared = 0
    for seed in range(block * 100, block * 100 + 100):
        l, keep = build(random.Random(seed))
        if not l.g.nodes:
            continue
        m = Machine(l, keep)
        got, steps = m.as_steps()
        assert got == m.in_order(), f"seed {seed}: {[len(s) for s in steps]}"
        shared += sum(len(s) > 1 for s in steps)
    assert shared > 50
