"""The reference's call sequences with every made tensor placed in one arena by
its lifetime, as a graph allocator does (a tensor's bytes are used again once
the last launch that reads it has run): the outputs' bits are those of the
same list over separate buffers."""
import pytest
import torch

from chatterbox_amdvulkan_amd import cbxops as C
from chatterbox_amdvulkan_amd.cfm_estimator import CFMEstimator
from chatterbox_amdvulkan_amd.flow_encoder import FlowEncoderCall
from chatterbox_amdvulkan_amd.hift_decode import HiFTDecode

pytestmark = pytest.mark.gpu


def place(g, keep):
    """Re-binds what the nodes make into one buffer, first fit over the planned
    launches; (the buffer, the tensors as they were)."""
    old = list(g._torch)
    key = [t.untyped_storage().data_ptr() for t in old]
    launch = {j: k for k, (_, f, n, _) in enumerate(g.plan(keep)) for j in range(f, f + n)}
    first, last = {}, {}
    for j, n in enumerate(g.nodes):
        if n.op != C.GOP_VIEW:
            first.setdefault(key[n.dst], launch[j])
        for i in (n.dst, *n.src):
            if i >= 0:
                last[key[i]] = launch[j]
    for i in keep:
        last[key[i]] = len(launch)
    size = {k: t.untyped_storage().nbytes() for k, t in zip(key, old)}
    live, at = [], {}
    for k in sorted(first, key=first.get):
        live = sorted(s for s in live if last[s[2]] >= first[k])
        need, lo = -(-size[k] // 256) * 256, 0
        for a, z, _ in live:
            if a - lo >= need:
                break
            lo = z
        at[k] = lo
        live.append((lo, lo + need, k))
    top = max(at[k] + size[k] for k in at)
    assert 3 * top < 2 * sum(size[k] for k in at)      # bytes are used again
    arena = torch.empty(top + 1024, dtype=torch.uint8, device="cuda")
    base = -arena.data_ptr() % 256
    for i, (t, k) in enumerate(zip(old, key)):
        if k in at:
            b = arena[base + at[k]:base + at[k] + size[k]].view(t.dtype)
            g.rebind(i, torch.as_strided(b, t.shape, t.stride(), b.storage_offset() + t.storage_offset()))
    return arena, old


@pytest.mark.parametrize("make", [lambda: HiFTDecode(100, seed=3), lambda: CFMEstimator(500, seed=3, n_mid=2, n_tr=2, mask_tail=40),
                                  lambda: FlowEncoderCall(125, seed=3, n_blocks=3, n_up_blocks=3)],
                         ids=["hift_decode", "cfm_estimator", "flow_encoder"])
def test_one_arena(cbx, make):
    e = make()
    g, keep = e.b.g, e.keep
    ex = g.capture(keep)
    ex.launch()
    torch.cuda.synchronize()
    ref = [g._torch[i].clone() for i in keep]
    ex.close()
    arena, old = place(g, keep)
    assert len(g.steps(keep)) < sum(p[0] != C.GL_VIEW for p in g.plan(keep))
    ex = g.capture(keep)
    for run in (ex.launch, ex.launch, lambda: g.compute(keep)):
        arena.fill_(255)
        run()
        torch.cuda.synchronize()
        for i, r in zip(keep, ref):
            assert torch.equal(g._torch[i], r), f"tensor {i}: {int((g._torch[i] != r).sum())} of {r.numel()} differ"
    ex.close()
    del old
    if hasattr(e, "close"):
        e.close()
