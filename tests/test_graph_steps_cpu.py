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
