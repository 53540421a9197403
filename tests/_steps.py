"""What a node list is issued as (Graph.steps) without a device: host tensors
at chosen addresses, and stand-ins for the prepared weights that the schedule
reads (their extents, never their data)."""
import ctypes

import torch

from chatterbox_amdvulkan_amd import cbxops as C
from chatterbox_amdvulkan_amd.ggml_nodes import NodeList

N_CU = 256


class WeightsHandle(ctypes.Structure):
    """struct cbx_conv1d_weights (cbx_api.cpp)."""
    _fields_ = [("serial", ctypes.c_uint64), ("device", ctypes.c_int), ("up", ctypes.c_int),
                ("k", ctypes.c_int64), ("taps", ctypes.c_int64), ("c_in", ctypes.c_int64), ("c_out", ctypes.c_int64),
                ("c_in_pad", ctypes.c_int64), ("c_out_pad", ctypes.c_int64), ("w_ph", ctypes.c_int64),
                ("data", ctypes.c_void_p)]


def handle(w: torch.Tensor) -> WeightsHandle:
    """The handle of conv1d weights made from w (C_out, C_in, K), device -1."""
    co, ci, k = w.shape
    return WeightsHandle(1, -1, 0, k, k, ci, co, ci, -(-co // 128) * 128, -(-co // 128) * 128 * k * ci, None)


class HostList(NodeList):
    """A node list over host memory that nothing reads or writes: every new
    tensor in address space of its own, or where `place` puts it."""

    def __init__(self):
        self.arena = torch.empty(0)
        self.handles = []
        super().__init__(lambda shape, dtype: self.empty(shape, dtype))

    @staticmethod
    def empty(shape, dtype=torch.float32):
        # rounded up to whole cache lines, so that no two tensors share one
        n = 1
        for s in shape:
            n *= s
        size = torch.empty(0, dtype=dtype).element_size()
        return torch.empty(-(-n * size // 64) * 64 // size + 64 // size, dtype=dtype)[:n].view(shape)

    def x(self, *shape):
        return self.t(self.empty(shape))

    def place(self, i: int, buf: torch.Tensor, off: int) -> int:
        """Tensor i at float `off` of buf."""
        t = self.at(i)
        self.g.rebind(i, buf[off:off + t.numel()].view(t.shape))
        return i

    def params(self, ch, K):
        p = {n + i: self.x(ch) for i in "12" for n in ("a", "ai", "b")}
        for i in "12":
            p["w" + i] = self.x(ch, ch, K)
        return p

    def conv_w(self, w: int) -> int:
        self.handles.append(handle(self.at(w)))
        return ctypes.addressof(self.handles[-1])

    def layer(self, x, ch, K, d):
        """A ResBlock layer; (its result, its first conv's output)."""
        p = self.params(ch, K)
        y = self.sublayer(x, p, d, self.conv_w(p["w1"]), self.conv_w(p["w2"]))
        sin = [i for i, n in enumerate(self.g.nodes) if n.op == C.GOP_UNARY and n.iparam == C.SIN][-1]
        return y, self.g.nodes[sin - 1].src[0]

    def steps(self, keep, n_cu=N_CU):
        return self.g.steps(keep, n_cu)


def kinds(g: C.Graph, keep, n_cu=N_CU):
    """The steps as lists of planned launch kinds."""
    plan = g.plan(keep)
    return [[plan[i][0] for i in s] for s in g.steps(keep, n_cu)]
