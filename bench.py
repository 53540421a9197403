"""Throughput of the fused layer-op path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu] [--quick]

Headline workload: the T3 prefill op chain -- gather of 512 token rows from
an [8194,1024] f32 table plus learned position rows 0..511 (one fused
kernel), LayerNorm+affine over [512,1024], tanh-GELU over [512,4096].  One
step = one pass of that chain.  Inputs are synthetic (seeded), resident in
HBM before the timed region; each step uses the next of several buffer sets
whose combined footprint exceeds twice the 256 MB Infinity Cache, so the
bytes come from HBM.  Steps are replayed from HIP graphs (captured once),
timed with events on the launch stream.

Prints ONE JSON line on stdout.  value = algorithmic bytes per step /
time per step (GB/s).  roofline = the dominant kernel (GELU), timed per
launch with HIP events.  cpu_baseline = the oracle (a C restatement of
ggml-cpu's arithmetic) running the same chain on the host.
"""
from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_HBM_GBS = 8000.0
MALL_DEFEAT_BYTES = 512 * 1024 * 1024


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=2000)
    ap.add_argument("--warmup", type=int, default=100)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    ap.add_argument("--cpu-seconds", type=float, default=10.0)
    ap.add_argument("--quick", action="store_true", help="skip the secondary workloads")
    ap.add_argument("--hift-conv", action="store_true",
                    help="only the HiFT conv1d / transposed-conv timings, as one JSON object (for profiling)")
    ap.add_argument("--only", choices=["decode", "serving", "cfm", "hift", "softmax", "t3_block", "t3_token", "hift_conv",
                                       "cfm_estimator", "hift_decode", "s3_encoder", "flow_encoder", "copy"],
                    help="run one secondary workload alone and print its JSON (no headline line)")
    ap.add_argument("--traffic-summary", nargs=2, metavar=("FETCH_DIR", "WRITE_DIR"),
                    help="print the markdown summary of two --pmc runs over --traffic-probe (no GPU)")
    ap.add_argument("--stats-summary", nargs=3, metavar=("STATS_DIR", "TITLE", "COMMAND"),
                    help="print the markdown summary of a --kernel-trace --stats run (no GPU)")
    ap.add_argument("--counters-summary", nargs="+", metavar="ARG",
                    help="TITLE COMMAND PMC_DIR [PMC_DIR ...]: markdown of --pmc runs over --traffic-probe (no GPU)")
    ap.add_argument("--traffic-probe", action="store_true",
                    help="only run the launches used by the FETCH_SIZE/WRITE_SIZE counter runs")
    return ap.parse_args()


# --------------------------------------------------------------------------- #
# prebuilt calls: descriptors are built once, launches are plain ctypes calls
# --------------------------------------------------------------------------- #

class PrefillSet:
    """Device buffers + descriptors of one T3-prefill step."""

    def __init__(self, C, W, torch, inp, f16_table=False):
        d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
        tab = inp["table"].astype(np.float16) if f16_table else inp["table"]
        self.t = {
            "table": d(tab), "ids": d(inp["ids"]), "pos_table": d(inp["pos_table"]), "pos_ids": d(inp["pos_ids"]),
            "ln_w": d(inp["ln_w"]), "ln_b": d(inp["ln_b"]), "ffn": d(inp["ffn"]),
        }
        self.t["h"] = torch.empty((W.N_PREFILL, W.D_MODEL), dtype=torch.float32, device="cuda")
        self.t["ln"] = torch.empty_like(self.t["h"])
        self.t["g"] = torch.empty_like(self.t["ffn"])
        self.d = {k: C.desc(v) for k, v in self.t.items()}
        self.r = {k: C.ctypes.byref(v) for k, v in self.d.items()}
        self.L = C.load()
        self.C = C

    def gather(self, s):
        r = self.r
        return self.L.cbx_get_rows_add(r["table"], r["ids"], r["pos_table"], r["pos_ids"], r["h"], s)

    def layer_norm(self, s):
        r = self.r
        return self.L.cbx_layer_norm(r["h"], r["ln_w"], r["ln_b"], 1e-5, -1, r["ln"], s)

    def embed_layer_norm(self, s):
        r = self.r
        return self.L.cbx_get_rows_add_layer_norm(r["table"], r["ids"], r["pos_table"], r["pos_ids"], r["ln_w"],
                                                  r["ln_b"], 1e-5, r["h"], r["ln"], s)

    def gelu(self, s):
        return self.L.cbx_gelu(self.r["ffn"], self.r["g"], s)

    def step(self, s):
        """Fused chain: token+position gather with LayerNorm, then GELU."""
        rc = self.embed_layer_norm(s) | self.gelu(s)
        if rc:
            raise self.C.CbxError(rc, self.C.last_error())

    def step_unfused(self, s):
        rc = self.gather(s) | self.layer_norm(s) | self.gelu(s)
        if rc:
            raise self.C.CbxError(rc, self.C.last_error())

    def step_one_launch(self, s):
        """The same two ops as one cbx_run_ops launch (their inputs are
        independent in this synthetic chain)."""
        if not hasattr(self, "batch"):
            C, t = self.C, self.t
            self.batch = C.OpBatch([
                C.Op(C.OP_GET_ROWS_ADD_LAYER_NORM, [t["table"], t["ids"], t["pos_table"], t["pos_ids"], t["ln_w"],
                                                    t["ln_b"]], [t["h"], t["ln"]], eps=1e-5),
                C.Op(C.OP_UNARY, [t["ffn"]], [t["g"]], act=C.GELU)])
        rc = self.L.cbx_run_ops(self.batch.arr, self.batch.n, s)
        if rc:
            raise self.C.CbxError(rc, self.C.last_error())


def cur_stream(torch):
    import ctypes

    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def capture(torch, fn):
    """HIP graph of fn(stream) captured through torch."""
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        fn(cur_stream(torch))
    return g


class StepGraphs:
    """HIP graphs that replay exactly `steps` steps over the buffer sets in
    order: whole rotations (one graph holding a step per set), then a graph
    of the first `steps mod n_sets` sets.  Every graph is replayed before
    anything is timed: a graph's first replay uploads it and costs several
    times a later one."""

    def __init__(self, torch, step_fns, steps):
        self.torch = torch
        self.full, rem = divmod(steps, len(step_fns))
        self.g_all = capture(torch, lambda s: [f(s) for f in step_fns]) if self.full else None
        self.g_rem = capture(torch, lambda s: [f(s) for f in step_fns[:rem]]) if rem else None

    def replay(self):
        for _ in range(self.full):
            self.g_all.replay()
        if self.g_rem is not None:
            self.g_rem.replay()

    def warm(self, warmup_steps, n_sets):
        """At least `warmup_steps` untimed steps, every graph replayed."""
        if self.g_all is not None:
            for _ in range(max(1, math.ceil(warmup_steps / n_sets))):
                self.g_all.replay()
        if self.g_rem is not None:
            self.g_rem.replay()
        self.torch.cuda.synchronize()

    def time_ms(self):
        """Milliseconds for the steps, events on the launch stream."""
        torch = self.torch
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        self.replay()
        e1.record()
        torch.cuda.synchronize()
        return e0.elapsed_time(e1)


def per_launch_ms(torch, fns, reps):
    """Average duration of one launch of a kernel in a back-to-back stream of
    its launches: one HIP graph holds a launch per buffer set (rotating
    inputs); it is replayed until `reps` launches have run, with events on
    the launch stream around the whole batch.  (An event pair around a
    single launch adds several microseconds of its own.)"""
    g = capture(torch, lambda s: [fn(s) for fn in fns])
    n_rep = max(1, reps // len(fns))
    g.replay()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(n_rep):
        g.replay()
    e1.record()
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / (n_rep * len(fns))
    del g
    return ms


# --------------------------------------------------------------------------- #
# workloads
# --------------------------------------------------------------------------- #

def same_bits(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint8), np.ascontiguousarray(b).view(np.uint8))


def bench_prefill(C, W, torch, steps, warmup, f16_table=False, fused=True, one_launch=False, resident=False):
    inp = W.prefill_inputs(f16_table=False)
    nbytes = W.prefill_bytes(f16_table, fused)
    per_step = sum(nbytes.values())
    # resident: every step reuses one buffer set (32 steps per graph), so the
    # bytes come from the Infinity Cache after the first step
    n_sets = 32 if resident else max(2, math.ceil(MALL_DEFEAT_BYTES / per_step))
    log(f"prefill{' f16' if f16_table else ''}{'' if fused else ' unfused'}{' one-launch' if one_launch else ''}"
        f"{' cache-resident' if resident else ''}: "
        f"{per_step} B/step, {n_sets} buffer sets")
    if resident:
        sets = [PrefillSet(C, W, torch, inp, f16_table)] * n_sets
    else:
        sets = [PrefillSet(C, W, torch, inp, f16_table) for _ in range(n_sets)]
    if one_launch:
        step = lambda st: st.step_one_launch  # noqa: E731
    else:
        step = (lambda st: st.step) if fused else (lambda st: st.step_unfused)

    # eager pass; the graph replays below must reproduce its results bit for
    # bit (parity with the CPU restatement is the test suite's job)
    for st in sets:
        step(st)(cur_stream(torch))
    torch.cuda.synchronize()
    eager = {k: sets[0].t[k].cpu().numpy() for k in ("h", "ln", "g")}
    for st in sets:
        for k in ("h", "ln", "g"):
            st.t[k].zero_()

    graphs = StepGraphs(torch, [step(st) for st in sets], steps)
    graphs.warm(warmup, n_sets)
    ms = graphs.time_ms()
    for k, v in eager.items():
        if not same_bits(sets[0].t[k].cpu().numpy(), v):
            raise SystemExit(f"bench: graph replay result {k} differs from the eager launch")

    reps = 400
    if one_launch:
        k_ms = {"run_ops": per_launch_ms(torch, [st.step_one_launch for st in sets], reps)}
    elif fused:
        k_ms = {"embed_layer_norm": per_launch_ms(torch, [st.embed_layer_norm for st in sets], reps),
                "gelu": per_launch_ms(torch, [st.gelu for st in sets], reps)}
    else:
        k_ms = {"gather_pos": per_launch_ms(torch, [st.gather for st in sets], reps),
                "layer_norm": per_launch_ms(torch, [st.layer_norm for st in sets], reps),
                "gelu": per_launch_ms(torch, [st.gelu for st in sets], reps)}
    del graphs, sets
    return {"ms_per_step": ms / steps, "bytes_per_step": per_step, "n_sets": n_sets,
            "kernel_ms": k_ms, "kernel_bytes": nbytes}


def dev_of(torch):
    return lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()


def time_steps_us(torch, fn, n_steps, reps=200):
    """Microseconds per step of fn(stream) (which runs n_steps steps),
    captured once as a HIP graph and replayed `reps` times."""
    g = capture(torch, fn)
    for _ in range(10):
        g.replay()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        g.replay()
    e1.record()
    torch.cuda.synchronize()
    us = e0.elapsed_time(e1) * 1000.0 / (reps * n_steps)
    del g
    return us


def check_rc(C, rc):
    if rc:
        raise C.CbxError(rc, C.last_error())


def bench_decode(C, W, torch):
    """T3 decode step (f32): RMSNorm+gamma [1,1024], RoPE q,k [1,16,64] at
    positions 0..29, SiLU(gate)*up [1,4096]; the 30 steps run from one HIP
    graph.  Three launch plans: one kernel per op (4 per step); q and k
    rotated by one launch (3 per step: the ops a real step can merge, since
    q and k come out of the same projection); all four in one launch."""
    d = dev_of(torch)
    L = C.load()
    cache = C.RopeCache(W.HEAD_DIM, mode=2, n_ctx_orig=2048, n_pos=2048)
    steps = []
    for s in range(W.DECODE_STEPS):
        t = {k: d(v) for k, v in W.decode_inputs(s).items()}
        t["y"] = torch.empty_like(t["x"])
        t["qo"], t["ko"], t["h"] = torch.empty_like(t["q"]), torch.empty_like(t["k"]), torch.empty_like(t["gate"])
        r = {k: C.ctypes.byref(C.desc(v)) for k, v in t.items()}
        qk = C.OpBatch([C.Op(C.OP_ROPE, [t["q"], t["pos"]], [t["qo"]], rope=cache),
                        C.Op(C.OP_ROPE, [t["k"], t["pos"]], [t["ko"]], rope=cache)])
        one = C.OpBatch([C.Op(C.OP_RMS_NORM, [t["x"], t["g"]], [t["y"]], eps=1e-5),
                         C.Op(C.OP_ROPE, [t["q"], t["pos"]], [t["qo"]], rope=cache),
                         C.Op(C.OP_ROPE, [t["k"], t["pos"]], [t["ko"]], rope=cache),
                         C.Op(C.OP_SWIGLU, [t["gate"], t["up"]], [t["h"]])])
        steps.append((t, r, qk, one))

    def per_op(s):
        for _, r, _, _ in steps:
            check_rc(C, L.cbx_rms_norm_mul(r["x"], r["g"], 1e-5, r["y"], s) |
                     L.cbx_rope_ext(r["q"], r["pos"], cache.handle, r["qo"], s) |
                     L.cbx_rope_ext(r["k"], r["pos"], cache.handle, r["ko"], s) |
                     L.cbx_swiglu(r["gate"], r["up"], r["h"], s))

    def qk_merged(s):
        for _, r, qk, _ in steps:
            check_rc(C, L.cbx_rms_norm_mul(r["x"], r["g"], 1e-5, r["y"], s) |
                     L.cbx_run_ops(qk.arr, qk.n, s) |
                     L.cbx_swiglu(r["gate"], r["up"], r["h"], s))

    def one_launch(s):
        for _, _, _, one in steps:
            check_rc(C, L.cbx_run_ops(one.arr, one.n, s))

    out = {}
    ref = None
    for name, fn in (("per_op_4_launches", per_op), ("qk_merged_3_launches", qk_merged),
                     ("one_launch", one_launch)):
        for t, *_ in steps:
            for k in ("y", "qo", "ko", "h"):
                t[k].zero_()
        fn(cur_stream(torch))
        torch.cuda.synchronize()
        got = [steps[-1][0][k].cpu().numpy() for k in ("y", "qo", "ko", "h")]
        if ref is None:
            ref = got
        elif not all(same_bits(a, b) for a, b in zip(got, ref)):
            raise SystemExit(f"bench: decode plan {name} differs from one kernel per op")
        out[name] = {"us_per_step": time_steps_us(torch, fn, W.DECODE_STEPS)}
    cache.close()
    nb = sum(W.decode_bytes().values())
    for v in out.values():
        v["GBps"] = nb / (v["us_per_step"] * 1e-6) / 1e9
    return dict(out, bytes_per_step=nb, note="30 steps' buffers stay cache resident (77,824 B per step)")


def bench_serving(C, W, torch, reps=400):
    """64-stream decode step, f16 storage: RMSNorm+gamma [64,1024], RoPE q,k
    [64,16,64] at per-stream positions, SiLU-gate [64,4096], Q8_0 gather of
    64 rows of [8194,1024] -- per op (5 launches) and as one launch, over
    rotating buffer sets larger than the Infinity Cache."""
    d = dev_of(torch)
    L = C.load()
    cache = C.RopeCache(W.HEAD_DIM, mode=2, n_ctx_orig=2048, n_pos=2048)
    base = {k: d(v) for k, v in W.serving_inputs().items()}
    nb = W.serving_bytes()
    per_step = sum(nb.values())
    n_sets = max(2, math.ceil(MALL_DEFEAT_BYTES / per_step))
    sets = []
    for _ in range(n_sets):
        t = {k: v.clone() for k, v in base.items()}
        t["y"], t["qo"], t["ko"] = torch.empty_like(t["x"]), torch.empty_like(t["q"]), torch.empty_like(t["k"])
        t["h"] = torch.empty_like(t["gate"])
        t["emb"] = torch.empty((W.N_STREAMS, W.D_MODEL), dtype=torch.float32, device="cuda")
        r = {k: C.ctypes.byref(C.desc(v, C.Q8_0 if k == "tab" else None)) for k, v in t.items()}
        one = C.OpBatch([C.Op(C.OP_RMS_NORM, [t["x"], t["g"]], [t["y"]], eps=1e-5),
                         C.Op(C.OP_ROPE, [t["q"], t["pos"]], [t["qo"]], rope=cache),
                         C.Op(C.OP_ROPE, [t["k"], t["pos"]], [t["ko"]], rope=cache),
                         C.Op(C.OP_SWIGLU, [t["gate"], t["up"]], [t["h"]]),
                         C.Op(C.OP_GET_ROWS, [t["tab"], t["ids"]], [t["emb"]], q8=[0])])
        sets.append((t, r, one))

    def per_op(st):
        _, r, _ = st
        return lambda s: check_rc(C, L.cbx_rms_norm_mul(r["x"], r["g"], 1e-5, r["y"], s) |
                                  L.cbx_rope_ext(r["q"], r["pos"], cache.handle, r["qo"], s) |
                                  L.cbx_rope_ext(r["k"], r["pos"], cache.handle, r["ko"], s) |
                                  L.cbx_swiglu(r["gate"], r["up"], r["h"], s) |
                                  L.cbx_get_rows(r["tab"], r["ids"], r["emb"], s))

    def one_launch(st):
        one = st[2]
        return lambda s: check_rc(C, L.cbx_run_ops(one.arr, one.n, s))

    out = {}
    ref = None
    for name, mk in (("per_op_5_launches", per_op), ("one_launch", one_launch)):
        fns = [mk(st) for st in sets]
        fns[0](cur_stream(torch))
        torch.cuda.synchronize()
        got = [sets[0][0][k].cpu().numpy() for k in ("y", "qo", "ko", "h", "emb")]
        if ref is None:
            ref = got
        elif not all(same_bits(a, b) for a, b in zip(got, ref)):
            raise SystemExit(f"bench: serving plan {name} differs from one kernel per op")
        us = per_launch_ms(torch, fns, reps) * 1000.0
        out[name] = {"us_per_step": us, "GBps": per_step / (us * 1e-6) / 1e9}
    # which op sets the one-launch time: each op alone as a one-op launch of
    # the same batch kernel (same bodies, same workgroup mapping)
    names = ("rms_norm_mul", "rope_q", "rope_k", "swiglu", "get_rows_q8_0")
    alone = {}
    for k, nm in enumerate(names):
        singles = []
        for t, _, one in sets:
            b1 = C.OpBatch([one.ops[k]])
            singles.append(b1)
        fns = [(lambda b1: lambda s: check_rc(C, L.cbx_run_ops(b1.arr, b1.n, s)))(b1) for b1 in singles]
        fns[0](cur_stream(torch))
        alone[nm] = per_launch_ms(torch, fns, reps) * 1000.0
    out["one_op_launch_us"] = alone
    cache.close()
    return dict(out, bytes_per_step=per_step, bytes=nb, buffer_sets=n_sets)


def bench_cfm(C, W, torch, reps=400):
    """CFM estimator ops of one flow step: GroupNorm(8)+affine+Mish on
    [2,256,500] and [2,512,500], LayerNorm+affine+NEOX RoPE (positions
    0..499) on [2,500,8x64] as one fused kernel (also timed as LayerNorm
    then RoPE); rotating buffer sets."""
    d = dev_of(torch)
    L = C.load()
    cache = C.RopeCache(W.HEAD_DIM, mode=2, n_ctx_orig=2048, n_pos=2048)
    base = {k: d(v) for k, v in W.cfm_inputs().items()}
    nb = W.cfm_bytes()
    per_step = sum(nb.values())
    n_sets = max(2, math.ceil(MALL_DEFEAT_BYTES / per_step))
    sets = []
    for _ in range(n_sets):
        t = {k: v.clone() for k, v in base.items()}
        for k in ("x256", "x512", "xa"):
            t["y" + k[1:]] = torch.empty_like(t[k])
        t["ya_rope"] = torch.empty_like(t["xa"])
        r = {k: C.ctypes.byref(C.desc(v)) for k, v in t.items()}
        ra = C.ctypes.byref(C.desc(t["ya"].view(2, W.CFM_T, W.CFM_HEADS, W.HEAD_DIM)))
        ro = C.ctypes.byref(C.desc(t["ya_rope"].view(2, W.CFM_T, W.CFM_HEADS, W.HEAD_DIM)))
        sets.append((t, r, ra, ro))

    ws = C.GroupNormWorkspace()

    def gn(key):
        """GroupNorm+affine+Mish with the statistics split over chunk
        workgroups (cbx_group_norm_ws; one workspace, stream-ordered)."""
        return lambda st: (lambda s: check_rc(C, L.cbx_group_norm_ws(st[1]["x" + key], W.CFM_GROUPS, 1e-5,
                                                                     st[1]["w" + key], st[1]["b" + key], C.MISH,
                                                                     st[1]["y" + key], ws.handle, s)))

    def gn_entry(key):
        """The same op through cbx_group_norm (the split over the library's
        scratch set for the stream)."""
        return lambda st: (lambda s: check_rc(C, L.cbx_group_norm(st[1]["x" + key], W.CFM_GROUPS, 1e-5,
                                                                  st[1]["w" + key], st[1]["b" + key], C.MISH,
                                                                  st[1]["y" + key], s)))

    def flow_batch(st):
        """The flow step's three ops in one launch (cbx_run_ops)."""
        t = st[0]
        b = C.OpBatch([C.Op(C.OP_GROUP_NORM, [t["x256"], t["w256"], t["b256"]], [t["y256"]], act=C.MISH, eps=1e-5,
                            iparam=W.CFM_GROUPS),
                       C.Op(C.OP_GROUP_NORM, [t["x512"], t["w512"], t["b512"]], [t["y512"]], act=C.MISH, eps=1e-5,
                            iparam=W.CFM_GROUPS),
                       C.Op(C.OP_LAYER_NORM_ROPE, [t["xa"], t["wa"], t["ba"], t["pos"]], [t["ya_rope"]], eps=1e-5,
                            rope=cache, iparam=W.HEAD_DIM)])
        return lambda s: b.launch(s)

    def ln(st):
        r = st[1]
        return lambda s: check_rc(C, L.cbx_layer_norm(r["xa"], r["wa"], r["ba"], 1e-5, -1, r["ya"], s))

    def rope(st):
        return lambda s: check_rc(C, L.cbx_rope_ext(st[2], st[1]["pos"], cache.handle, st[3], s))

    def ln_rope(st):
        r = st[1]
        return lambda s: check_rc(C, L.cbx_layer_norm_rope(r["xa"], r["wa"], r["ba"], 1e-5, W.HEAD_DIM, r["pos"],
                                                           cache.handle, r["ya_rope"], s))

    out = {}
    for name, mk in (("group_norm_mish_256", gn("256")), ("group_norm_mish_512", gn("512")),
                     ("group_norm_mish_256_entry_point", gn_entry("256")),
                     ("group_norm_mish_512_entry_point", gn_entry("512")),
                     ("layer_norm_1024x512", ln), ("rope_2x500x8x64", rope), ("layer_norm_rope_fused", ln_rope)):
        fns = [mk(st) for st in sets]
        for f in fns:
            f(cur_stream(torch))
        out[name] = {"us": per_launch_ms(torch, fns, reps) * 1000.0}
    # the fused kernel must reproduce layer_norm then rope_ext bit for bit
    torch.cuda.synchronize()
    fused = sets[0][0]["ya_rope"].cpu().numpy()
    for f in (ln(sets[0]), rope(sets[0])):
        f(cur_stream(torch))
    torch.cuda.synchronize()
    if not same_bits(fused, sets[0][0]["ya_rope"].cpu().numpy()):
        raise SystemExit("bench: fused LayerNorm+RoPE differs from LayerNorm then RoPE")
    step = lambda st: (lambda s: [mk(st)(s) for mk in (gn("256"), gn("512"), ln_rope)])  # noqa: E731
    out["flow_step"] = {"us": per_launch_ms(torch, [step(st) for st in sets], reps) * 1000.0,
                        "launches": "group_norm+mish [2,256,500], group_norm+mish [2,512,500], "
                                    "layer_norm_rope [2,500,512]"}
    # the three ops in one launch must give the three launches' bits
    t0 = sets[0][0]
    step(sets[0])(cur_stream(torch))
    torch.cuda.synchronize()
    three = [t0[k].cpu().numpy() for k in ("y256", "y512", "ya_rope")]
    for k in ("y256", "y512", "ya_rope"):
        t0[k].fill_(float("nan"))
    flows = [flow_batch(st) for st in sets]
    flows[0](cur_stream(torch))
    torch.cuda.synchronize()
    for k, ref in zip(("y256", "y512", "ya_rope"), three):
        if not same_bits(ref, t0[k].cpu().numpy()):
            raise SystemExit(f"bench: the one-launch flow step's {k} differs from the three launches'")
    out["flow_step_one_launch"] = {"us": per_launch_ms(torch, flows, reps) * 1000.0,
                                   "launches": "cbx_run_ops: both group norms (split) + layer_norm_rope"}
    for k in ("group_norm_mish_256", "group_norm_mish_512"):
        out[k]["GBps"] = nb[k] / (out[k]["us"] * 1e-6) / 1e9
        out[k + "_entry_point"]["GBps"] = nb[k] / (out[k + "_entry_point"]["us"] * 1e-6) / 1e9
    # the workspace form and the entry point must give the same bits
    for key in ("256", "512"):
        gn(key)(sets[0])(cur_stream(torch))
        torch.cuda.synchronize()
        split = t0["y" + key].cpu().numpy()
        gn_entry(key)(sets[0])(cur_stream(torch))
        torch.cuda.synchronize()
        if not same_bits(split, t0["y" + key].cpu().numpy()):
            raise SystemExit(f"bench: GroupNorm [2,{key},500] differs between cbx_group_norm_ws and cbx_group_norm")
    out["layer_norm_rope_fused"]["GBps"] = nb["layer_norm_rope"] / (out["layer_norm_rope_fused"]["us"] * 1e-6) / 1e9
    lr = out["layer_norm_1024x512"]["us"] + out["rope_2x500x8x64"]["us"]
    out["layer_norm_then_rope_GBps_vs_fused_bytes"] = nb["layer_norm_rope"] / (lr * 1e-6) / 1e9
    out["flow_step"]["GBps"] = per_step / (out["flow_step"]["us"] * 1e-6) / 1e9
    out["flow_step_one_launch"]["GBps"] = per_step / (out["flow_step_one_launch"]["us"] * 1e-6) / 1e9
    cache.close()
    ws.close()
    return dict(out, bytes_per_flow_step=per_step, bytes=nb, buffer_sets=n_sets)


def bench_softmax(C, W, torch, reps=200):
    """Attention-score epilogue (scale -> diag_mask_inf -> soft_max, one
    kernel): T3 prefill scores [16 heads, 512, 512] with the causal mask, and
    CFM scores [2, 8 heads, 500, 500] without; rotating buffer sets."""
    L = C.load()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(W.seed_of(6, 0))
    out = {}
    for name, shape, sc, n_past in (("t3_prefill_causal_16x512x512", (16, 512, 512), 0.125, 0),
                                    ("cfm_2x8x500x500", (2, 8, 500, 500), 0.125, -1)):
        n = int(np.prod(shape))
        per = 8 * n
        n_sets = max(2, math.ceil(MALL_DEFEAT_BYTES / per))
        xs = [torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, 4.0, generator=gen)
              for _ in range(n_sets)]
        ys = [torch.empty_like(x) for x in xs]
        rx = [C.ctypes.byref(C.desc(x)) for x in xs]
        ry = [C.ctypes.byref(C.desc(y)) for y in ys]
        fns = [(lambda i: lambda s: check_rc(C, L.cbx_scale_diag_mask_soft_max(rx[i], sc, n_past, ry[i], s)))(i)
               for i in range(n_sets)]
        for f in fns:
            f(cur_stream(torch))
        ms = per_launch_ms(torch, fns, reps)
        out[name] = {"us": ms * 1000.0, "bytes": per, "GBps": per / (ms * 1e-3) / 1e9, "buffer_sets": n_sets}
        del xs, ys
    return out


def graph_exec_costs(C, torch, base, n_blocks, s, calls=100):
    """Host and device microseconds per call of cbx_graph_compute and of
    cbx_graph_exec_launch on `n_blocks` T3 blocks' element-wise node lists
    (3 launches each), each block writing its own intermediates."""
    import ctypes

    L = C.load()
    N, D = base["h"].shape
    F = base["fc_mm"].shape[1]
    g = C.Graph()
    T = {k: g.tensor(v) for k, v in base.items()}
    keep = []
    for _ in range(n_blocks):
        t = {k: g.tensor(torch.empty((N, D), dtype=torch.float32, device="cuda"))
             for k in ("cur", "res", "n", "m", "ln2", "pcur", "h2", "n2", "m2", "ln1")}
        t.update({k: g.tensor(torch.empty((N, F), dtype=torch.float32, device="cuda")) for k in ("fcb", "gelu")})
        g.node(C.GOP_ADD, t["cur"], (T["attn_mm"], T["out_b"]))
        g.node(C.GOP_ADD, t["res"], (t["cur"], T["h"]))
        g.node(C.GOP_NORM, t["n"], (t["res"],), fparam=1e-5)
        g.node(C.GOP_MUL, t["m"], (t["n"], T["ln2_w"]))
        g.node(C.GOP_ADD, t["ln2"], (t["m"], T["ln2_b"]))
        g.node(C.GOP_ADD, t["fcb"], (T["fc_mm"], T["fc_b"]))
        g.node(C.GOP_UNARY, t["gelu"], (t["fcb"],), iparam=C.GELU)
        g.node(C.GOP_ADD, t["pcur"], (T["proj_mm"], T["proj_b"]))
        g.node(C.GOP_ADD, t["h2"], (t["pcur"], t["res"]))
        g.node(C.GOP_NORM, t["n2"], (t["h2"],), fparam=1e-5)
        g.node(C.GOP_MUL, t["m2"], (t["n2"], T["ln1_w"]))
        g.node(C.GOP_ADD, t["ln1"], (t["m2"], T["ln1_b"]))
        keep += [t["ln2"], t["gelu"], t["h2"], t["ln1"]]
    Tn, Nn, Kn = g._arrays(keep)
    n = ctypes.c_int32(0)
    ex = g.capture(keep)

    def compute():
        check_rc(C, L.cbx_graph_compute(Tn, len(g._descs), Nn, len(g.nodes), Kn, len(keep), s, ctypes.byref(n)))

    res = {"launches": ex.n_launches, "kernels": len(g.steps(keep))}
    for name, f in (("compute", compute), ("exec", lambda: ex.launch(s))):
        for _ in range(5):
            f()
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        tm = time.perf_counter()
        e0.record()
        for _ in range(calls):
            f()
        host = (time.perf_counter() - tm) / calls * 1e6
        e1.record()
        torch.cuda.synchronize()
        res[name] = {"host_us": host, "device_us": e0.elapsed_time(e1) * 1000.0 / calls}
    # re-pointing the exec at the list with other buffers for a matmul's output
    # (the next step of a loop: the same launches, taken in place) against
    # capturing anew; three in turn, so that neither of the exec's two
    # instantiations holds the next one already
    bufs = [base["fc_mm"], torch.empty_like(base["fc_mm"]), torch.empty_like(base["fc_mm"])]
    ip = ctypes.c_int32(0)
    upd = new = 0.0
    reps = max(1, calls // 5)
    for k in range(reps):
        Tn[T["fc_mm"]].data = bufs[(k + 1) % 3].data_ptr()
        torch.cuda.synchronize()
        tm = time.perf_counter()
        check_rc(C, L.cbx_graph_exec_update(ex.handle, Tn, len(g._descs), Nn, len(g.nodes), Kn, len(keep),
                                            ctypes.byref(n), ctypes.byref(ip)))
        upd += time.perf_counter() - tm
        ex.launch(s)
        h2 = ctypes.c_void_p()
        tm = time.perf_counter()
        check_rc(C, L.cbx_graph_exec_create(Tn, len(g._descs), Nn, len(g.nodes), Kn, len(keep), ctypes.byref(h2),
                                            ctypes.byref(n)))
        new += time.perf_counter() - tm
        L.cbx_graph_exec_destroy(h2)
    res["update_host_us"] = upd / reps * 1e6
    res["update_in_place"] = bool(ip.value)
    res["create_host_us"] = new / reps * 1e6
    ex.close()
    return res


def bench_t3_block(C, W, torch, reps=300):
    """One T3 block's element-wise nodes at prefill size [512,1024] /
    [512,4096] (t3.cpp:526-546; the matmul outputs given): the residual join
    + pre-FFN LayerNorm, fc bias + GELU, and the projection's residual join +
    the next block's LayerNorm -- three launches planned from the ggml node
    list by cbx_graph_plan, then issued with cbx_graph_launch over rotating
    buffer sets.  Also the host cost of cbx_graph_compute on that list."""
    d = dev_of(torch)
    L = C.load()
    base = {k: d(v) for k, v in W.t3_block_inputs().items()}
    nb = W.t3_block_bytes()
    per_step = nb["residual_ln2"] + nb["fc_bias_gelu"] + nb["residual_next_ln1"]
    n_sets = max(2, math.ceil(MALL_DEFEAT_BYTES / per_step))
    N, D, F = W.N_PREFILL, W.D_MODEL, W.D_FF

    def graph_of(t):
        g = C.Graph()
        T = {k: g.tensor(v) for k, v in t.items()}
        g.node(C.GOP_ADD, T["cur"], (T["attn_mm"], T["out_b"]))
        g.node(C.GOP_ADD, T["res"], (T["cur"], T["h"]))
        g.node(C.GOP_NORM, T["n"], (T["res"],), fparam=1e-5)
        g.node(C.GOP_MUL, T["m"], (T["n"], T["ln2_w"]))
        g.node(C.GOP_ADD, T["ln2"], (T["m"], T["ln2_b"]))
        g.node(C.GOP_ADD, T["fcb"], (T["fc_mm"], T["fc_b"]))
        g.node(C.GOP_UNARY, T["gelu"], (T["fcb"],), iparam=C.GELU)
        g.node(C.GOP_ADD, T["pcur"], (T["proj_mm"], T["proj_b"]))
        g.node(C.GOP_ADD, T["h2"], (T["pcur"], T["res"]))
        g.node(C.GOP_NORM, T["n2"], (T["h2"],), fparam=1e-5)
        g.node(C.GOP_MUL, T["m2"], (T["n2"], T["ln1_w"]))
        g.node(C.GOP_ADD, T["ln1"], (T["m2"], T["ln1_b"]))
        keep = [T["ln2"], T["gelu"], T["h2"], T["ln1"]]
        plan = g.plan(keep)
        arrs = g._arrays(keep)
        return g, plan, arrs, keep

    sets = []
    for _ in range(n_sets):
        t = {k: v.clone() for k, v in base.items()}
        for k in ("cur", "res", "n", "m", "ln2", "pcur", "h2", "n2", "m2", "ln1"):
            t[k] = torch.empty((N, D), dtype=torch.float32, device="cuda")
        for k in ("fcb", "gelu"):
            t[k] = torch.empty((N, F), dtype=torch.float32, device="cuda")
        g, plan, arrs, keep = graph_of(t)
        launches = [C.GLaunch(*p) for p in plan]
        sets.append((t, g, plan, arrs, launches, keep))
    kinds = [p[0] for p in sets[0][2]]
    if kinds != [C.GL_ADD_LAYER_NORM, C.GL_BIAS_ACT, C.GL_ADD_LAYER_NORM]:
        raise SystemExit(f"bench: unexpected T3 block plan {kinds}")

    def one(st, k):
        _, g, _, (Tn, Nn, _), launches, _ = st
        nt, nn = len(g._descs), len(g.nodes)
        lr = C.ctypes.byref(launches[k])
        return lambda s: check_rc(C, L.cbx_graph_launch(Tn, nt, Nn, nn, lr, s))

    out = {}
    for name, k in (("residual_ln2", 0), ("fc_bias_gelu", 1), ("residual_next_ln1", 2)):
        fns = [one(st, k) for st in sets]
        for f in fns:
            f(cur_stream(torch))
        us = per_launch_ms(torch, fns, reps) * 1000.0
        out[name] = {"us": us, "bytes": nb[name], "GBps": nb[name] / (us * 1e-6) / 1e9}
    block = [(lambda st: lambda s: [one(st, k)(s) for k in range(3)])(st) for st in sets]
    us = per_launch_ms(torch, block, reps) * 1000.0
    out["block"] = {"us": us, "launches": 3, "bytes": per_step, "GBps": per_step / (us * 1e-6) / 1e9,
                    "ggml_node_bytes": nb["ggml_nodes"],
                    "ggml_node_bytes_ratio": nb["ggml_nodes"] / per_step}
    # host cost of planning + issuing the whole list (no GPU sync inside)
    t0 = sets[0]
    Tn, Nn, Kn = t0[3]
    n = C.ctypes.c_int32(0)
    s = cur_stream(torch)
    torch.cuda.synchronize()
    tm = time.perf_counter()
    for _ in range(200):
        check_rc(C, L.cbx_graph_compute(Tn, len(t0[1]._descs), Nn, len(t0[1].nodes), Kn, len(t0[5]), s,
                                        C.ctypes.byref(n)))
    host_us = (time.perf_counter() - tm) / 200 * 1e6
    torch.cuda.synchronize()
    out["graph_compute_host_us_per_call"] = host_us
    # host cost per call of cbx_graph_compute (plans and launches every
    # call) against cbx_graph_exec_launch (the list captured once into a HIP
    # graph), for the block's list and for 16 blocks' lists in one (48
    # launches; the blocks share the inputs), with the device time per call
    # of the same back-to-back calls (inputs cache-resident)
    out["graph_exec"] = {f"{nb}_blocks": graph_exec_costs(C, torch, base, nb, s) for nb in (1, 16)}
    return dict(out, buffer_sets=n_sets)


def bench_t3_token(C, W, torch, reps=200, tokens=64):
    """One T3 decode step's element-wise nodes at N_new = 1 (t3.cpp:446-546:
    the input embedding, 24 blocks' LN-1, qkv bias, score softmax, residual
    joins with LN-2 and the next LN-1, fc bias + GELU, the final LN; the
    matmul outputs given), planned into 121 launches by the node-list
    executor.  Device time per token from back-to-back replays of the list
    captured into a HIP graph (cbx_graph_exec); the same list planned and
    launched every token (cbx_graph_compute); and a decode loop of `tokens`
    consecutive tokens, each re-pointed with cbx_graph_exec_update (the
    scores one column longer, the mask's n_past), its token and position
    written, then replayed -- wall time per token, host time of the update."""
    from chatterbox_amdvulkan_amd import t3_decode as T

    inp = W.t3_token_inputs()
    dev = T.upload(inp)
    n0 = 255
    st = T.T3DecodeStep(dev, n0)
    st.set_token(17, n0)
    ex = st.graph.capture(st.keep)
    s = cur_stream(torch)
    out = {"launches": ex.n_launches, "kernels": len(st.graph.steps(st.keep)), "blocks": st.n_blocks, "n_past": n0,
           "bytes_per_token": W.t3_token_bytes(st.n_blocks, n0)}
    for _ in range(10):
        ex.launch(s)
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        ex.launch(s)
    e1.record()
    torch.cuda.synchronize()
    dev_us = e0.elapsed_time(e1) * 1000.0 / reps
    out["exec_replay_us_per_token"] = dev_us
    out["exec_replay_us_per_kernel"] = dev_us / out["kernels"]
    # plan + launch every token (no graph)
    for _ in range(3):
        st.graph.compute(st.keep)
    torch.cuda.synchronize()
    n_c = max(20, reps // 4)
    tm = time.perf_counter()
    e0.record()
    for _ in range(n_c):
        st.graph.compute(st.keep)
    host = (time.perf_counter() - tm) / n_c * 1e6
    e1.record()
    torch.cuda.synchronize()
    out["graph_compute_us_per_token"] = {"host_us": host, "device_us": e0.elapsed_time(e1) * 1000.0 / n_c}
    # a decode loop: update + token write + replay per token, no sync inside
    upd = 0.0
    torch.cuda.synchronize()
    t_loop = time.perf_counter()
    for t in range(tokens):
        n_past = n0 + 1 + t
        st.retarget(n_past)
        tm = time.perf_counter()
        ok = ex.update(st.graph, st.keep)
        upd += time.perf_counter() - tm
        if not ok:
            raise SystemExit("bench: the T3 token list was not updated in place")
        st.set_token((17 * t) % W.T3_SPEECH_VOCAB, n_past)
        ex.launch(s)
    torch.cuda.synchronize()
    out["decode_loop_us_per_token"] = (time.perf_counter() - t_loop) / tokens * 1e6
    out["update_host_us_per_token"] = upd / tokens * 1e6
    out["decode_loop_tokens"] = tokens
    ex.close()
    return out


def estimator_bytes(C, e, plan):
    """Bytes one node-list call's launches move: per launch, every tensor it
    reads from outside the launch once (a causal conv's weights as their
    prepared f16 copy, a gather's table as the rows it gathers) and every
    tensor it stores (the last node's, the stored residual sum, the first
    of two outputs)."""
    nd, at = e.graph.nodes, e.b.at
    total = 0
    for kind, f, n, flags in plan:
        if kind == C.GL_VIEW:
            continue
        made = {nd[j].dst for j in range(f, f + n)}
        reads = {s for j in range(f, f + n) for s in nd[j].src if s >= 0} - made
        if kind == C.GL_CAUSAL_CONV1D:
            w = nd[f + 7].src[0]          # the weight tensor of the im2col node
            reads.discard(w)
            total += at(w).numel() * 2
        if kind == C.GL_GET_ROWS:         # the gathered rows, not the whole table
            reads.discard(nd[f].src[0])
            total += at(nd[f].dst).numel() * at(nd[f].dst).element_size()
        total += sum(at(s).numel() * at(s).element_size() for s in reads)
        y = at(nd[f + n - 1].dst)
        total += y.numel() * y.element_size()
        if kind == C.GL_ADD_LAYER_NORM and not flags & 1:
            total += y.numel() * y.element_size()   # the residual sum, stored too
        if kind in (C.GL_BIAS_ADD_TWO, C.GL_ROPE_TWO, C.GL_BIAS_ADD_PAIR):   # two outputs: the other one
            k = f if kind != C.GL_BIAS_ADD_PAIR else next(j for j in range(f + 2, f + n) if nd[j].op == C.GOP_ADD)
            total += at(nd[k].dst).numel() * at(nd[k].dst).element_size()
    return total


def bench_cfm_estimator(C, torch, T=500, reps=20):
    """One CFM estimator call's element-wise nodes (cfm_decoder.cpp:395-558:
    14 resnet blocks with their 29 causal blocks, 56 transformer blocks; the
    matmul outputs given, the causal convs on the library's conv kernel) at
    the reference's sizes over T frames, planned into one list of launches
    (chatterbox_amdvulkan_amd/cfm_estimator.py).  Device time per call from
    back-to-back replays of the list captured into a HIP graph
    (cbx_graph_exec), and the same list planned and launched each call
    (cbx_graph_compute)."""
    from chatterbox_amdvulkan_amd.cfm_estimator import CFMEstimator

    e = CFMEstimator(T, seed=5)
    try:
        plan = e.plan()
        ex = e.graph.capture(e.keep)
        s = cur_stream(torch)
        nbytes = estimator_bytes(C, e, plan)
        kinds = {}
        names = {v: k[3:].lower() for k, v in vars(C).items() if k.startswith("GL_") and isinstance(v, int)}
        for p in plan:
            if p[0] != C.GL_VIEW:
                kinds[names[p[0]]] = kinds.get(names[p[0]], 0) + 1
        out = {"reference_sequence": f"cfm_decoder.cpp:395-558, T_mel {T}, 14 resnet blocks, 56 transformer blocks",
               "launches": ex.n_launches, "kernels": len(e.graph.steps(e.keep)), "launches_by_kind": kinds,
               "bytes_per_call": nbytes}
        for _ in range(3):
            ex.launch(s)
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(reps):
            ex.launch(s)
        e1.record()
        torch.cuda.synchronize()
        dev_us = e0.elapsed_time(e1) * 1000.0 / reps
        out["exec_replay_us_per_call"] = dev_us
        out["exec_replay_us_per_kernel"] = dev_us / out["kernels"]
        out["GBps"] = nbytes / (dev_us * 1e-6) / 1e9
        ex.close()
        for _ in range(2):
            e.graph.compute(e.keep)
        torch.cuda.synchronize()
        n_c = max(5, reps // 4)
        tm = time.perf_counter()
        e0.record()
        for _ in range(n_c):
            e.graph.compute(e.keep)
        host = (time.perf_counter() - tm) / n_c * 1e6
        e1.record()
        torch.cuda.synchronize()
        out["graph_compute_us_per_call"] = {"host_us": host, "device_us": e0.elapsed_time(e1) * 1000.0 / n_c}
        return out
    finally:
        e.close()


def bench_node_list(C, torch, e, ref, reps):
    """Device time per call of a reference-sequence node list e (its graph,
    keep list and plan) from back-to-back replays of the list captured into
    a HIP graph (cbx_graph_exec), and the same list planned and launched each
    call (cbx_graph_compute)."""
    plan = e.plan()
    ex = e.graph.capture(e.keep)
    s = cur_stream(torch)
    nbytes = estimator_bytes(C, e, plan)
    kinds = {}
    names = {v: k[3:].lower() for k, v in vars(C).items() if k.startswith("GL_") and isinstance(v, int)}
    for p in plan:
        if p[0] != C.GL_VIEW:
            kinds[names[p[0]]] = kinds.get(names[p[0]], 0) + 1
    out = {"reference_sequence": ref, "launches": ex.n_launches, "kernels": len(e.graph.steps(e.keep)),
           "launches_by_kind": kinds, "bytes_per_call": nbytes}
    for _ in range(3):
        ex.launch(s)
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        ex.launch(s)
    e1.record()
    torch.cuda.synchronize()
    dev_us = e0.elapsed_time(e1) * 1000.0 / reps
    out["exec_replay_us_per_call"] = dev_us
    out["exec_replay_us_per_kernel"] = dev_us / out["kernels"]
    out["GBps"] = nbytes / (dev_us * 1e-6) / 1e9
    ex.close()
    for _ in range(2):
        e.graph.compute(e.keep)
    torch.cuda.synchronize()
    n_c = max(5, reps // 4)
    tm = time.perf_counter()
    e0.record()
    for _ in range(n_c):
        e.graph.compute(e.keep)
    host = (time.perf_counter() - tm) / n_c * 1e6
    e1.record()
    torch.cuda.synchronize()
    out["graph_compute_us_per_call"] = {"host_us": host, "device_us": e0.elapsed_time(e1) * 1000.0 / n_c}
    return out


def bench_s3_encoder(C, torch, T_mel=1000, reps=20):
    """One S3 speech-tokenizer encoder call's element-wise nodes
    (s3enc.cpp:124-290: the front convs' bias + GELU-erf, 6 layers' LayerNorms,
    q / k RoPE, FSMN join, score softmax, bias + residual joins, bias +
    GELU-erf; matmul, conv and FSMN outputs given) over T_mel mel frames,
    planned into one list of launches (chatterbox_amdvulkan_amd/
    s3_encoder.py)."""
    from chatterbox_amdvulkan_amd.s3_encoder import S3EncoderCall

    e = S3EncoderCall(T_mel, seed=5)
    try:
        return bench_node_list(C, torch, e, f"s3enc.cpp:124-290, T_mel {T_mel} ({e.T_tok} tokens), "
                               f"{e.n_layer} layers", reps)
    finally:
        e.close()


def bench_flow_encoder(C, torch, T=250, reps=20):
    """One flow-encoder call's element-wise nodes (flow_encoder.cpp:537-700:
    the speech-token gather, the embed linears' bias + LayerNorm + scale, the
    pre-lookahead's bias + LeakyReLU and residual, 6 + 4 conformer blocks'
    bias adds, pos_bias adds, score softmax, bias + residual + LayerNorm
    joins and bias + SiLU, after_norm, encoder_proj's bias; matmul, conv and
    layout outputs given) over T speech tokens, planned into one list of
    launches (chatterbox_amdvulkan_amd/flow_encoder.py)."""
    from chatterbox_amdvulkan_amd.flow_encoder import FlowEncoderCall

    e = FlowEncoderCall(T, seed=6)
    return bench_node_list(C, torch, e, f"flow_encoder.cpp:537-700, {T} tokens ({2 * T} frames), "
                           f"{e.n_blocks} + {e.n_up_blocks} blocks", reps)


def bench_hift_decode(C, torch, T_mel=500, reps=10):
    """One HiFT vocoder decode (hift_vocoder.cpp:613-749: conv_pre, the three
    upsampling stages with their source convs and resblocks, conv_post; the
    host STFT of the source and the iSTFT left out) over T_mel mel frames,
    planned into one list of launches (chatterbox_amdvulkan_amd/
    hift_decode.py).  Device time per decode from back-to-back replays of
    the list captured into a HIP graph (cbx_graph_exec), the convs'
    arithmetic rate against the f16 MFMA peak, and the same list planned and
    launched each decode (cbx_graph_compute)."""
    from chatterbox_amdvulkan_amd.hift_decode import HiFTDecode

    e = HiFTDecode(T_mel, seed=5)
    try:
        plan = e.plan()
        ex = e.graph.capture(e.keep)
        s = cur_stream(torch)
        flops = e.flops()
        kinds = {}
        names = {v: k[3:].lower() for k, v in vars(C).items() if k.startswith("GL_") and isinstance(v, int)}
        for p in plan:
            if p[0] != C.GL_VIEW:
                kinds[names[p[0]]] = kinds.get(names[p[0]], 0) + 1
        out = {"reference_sequence": f"hift_vocoder.cpp:613-749, T_mel {T_mel} "
                                     f"(stages of {e.stage_frames[0]}, {e.stage_frames[1]}, {e.stage_frames[2]} frames)",
               "launches": ex.n_launches, "kernels": len(e.graph.steps(e.keep)), "launches_by_kind": kinds,
               "conv_flop_per_decode": flops}
        for _ in range(2):
            ex.launch(s)
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(reps):
            ex.launch(s)
        e1.record()
        torch.cuda.synchronize()
        dev_us = e0.elapsed_time(e1) * 1000.0 / reps
        out["exec_replay_us_per_decode"] = dev_us
        out["conv_TFLOPs"] = flops / (dev_us * 1e-6) / 1e12
        out["pct_of_f16_mfma_peak"] = 100.0 * out["conv_TFLOPs"] / PEAK_MFMA_F16_TFLOPS
        out["audio_seconds_per_decode"] = T_mel * 480 / 24000
        ex.close()
        e.graph.compute(e.keep)
        torch.cuda.synchronize()
        n_c = max(3, reps // 2)
        tm = time.perf_counter()
        e0.record()
        for _ in range(n_c):
            e.graph.compute(e.keep)
        host = (time.perf_counter() - tm) / n_c * 1e6
        e1.record()
        torch.cuda.synchronize()
        out["graph_compute_us_per_decode"] = {"host_us": host, "device_us": e0.elapsed_time(e1) * 1000.0 / n_c}
        return out
    finally:
        e.close()


PEAK_MFMA_F16_TFLOPS = 2500.0


def bench_hift_conv(C, W, torch, reps=60):
    """HiFT ResBlock convs (hift_vocoder.cpp:119-138) at the vocoder stage
    shapes [1,256,6000], [1,128,48000], [1,64,120000]: snake -> conv1d
    (K 11, dilation 5) + bias, snake -> conv1d (K 3, dilation 1) + bias + x,
    and one whole sublayer (snake -> conv K 11 d 5 -> snake -> conv K 11 d 1
    -> + x, two launches); then the three upsamplers.  f16 operands, f32
    accumulation on the matrix cores; algorithmic FLOPs 2*C_in*C_out*K*T_out
    per conv.  Launches rotate over buffer sets whose combined size exceeds
    twice the Infinity Cache, so activations come from HBM."""
    d = dev_of(torch)
    L = C.load()
    out = {}

    def sets_for(nbytes):
        return max(2, math.ceil(MALL_DEFEAT_BYTES / nbytes))

    def rate(flops, nbytes, us, **kw):
        return dict({"us": us, "TFLOPs": flops / (us * 1e-6) / 1e12,
                     "pct_of_mfma_f16_peak": 100.0 * flops / (us * 1e-6) / 1e12 / PEAK_MFMA_F16_TFLOPS,
                     "GBps": nbytes / (us * 1e-6) / 1e9}, **kw)

    for (Ch, T) in ((256, 6000), (128, 48000), (64, 120000)):
        n_sets = sets_for(3 * 4 * T * Ch)
        x0 = d(W.normal(W.seed_of(8, Ch), (T, Ch)))
        bufs = [{"x": x0 if i == 0 else x0.clone(), "h": torch.empty_like(x0), "y": torch.empty_like(x0)}
                for i in range(n_sets)]
        a, ai = (d(v) for v in W.snake_alpha(Ch, 3))
        bias = d(W.normal(W.seed_of(8, Ch + 1), (Ch,), 0.0, 0.1))
        ws = {K: C.Conv1dWeights(d(W.normal(W.seed_of(8, Ch + K), (Ch, Ch, K), 0.0, 1.0 / np.sqrt(Ch * K))))
              for K in (3, 11)}
        Rc = {k: C.ctypes.byref(C.desc(v)) for k, v in dict(a=a, ai=ai, b=bias).items()}
        Rs = [{k: C.ctypes.byref(C.desc(v)) for k, v in b.items()} for b in bufs]
        res = {"buffer_sets": n_sets}

        def conv(R, K, dil, src, dst, residual):
            pad = (K - 1) // 2 * dil
            return lambda s: check_rc(C, L.cbx_conv1d(R[src], ws[K].handle, 1, pad, dil, C.CONV_PRO_SNAKE, Rc["a"],
                                                      Rc["ai"], 0.0, Rc["b"], R["x"] if residual else None, R[dst],
                                                      s))
        for name, K, dil, residual in (("k11_d5", 11, 5, False), ("k3_d1_residual", 3, 1, True)):
            fns = [conv(R, K, dil, "x", "y", residual) for R in Rs]
            fns[0](cur_stream(torch))
            us = per_launch_ms(torch, fns, max(reps, 2 * n_sets)) * 1000.0
            res[name] = rate(2.0 * Ch * Ch * K * T, 4 * T * Ch * (3 if residual else 2), us)
        subs = []
        for R in Rs:
            c1, c2 = conv(R, 11, 5, "x", "h", False), conv(R, 11, 1, "h", "y", True)
            subs.append(lambda s, c1=c1, c2=c2: (c1(s), c2(s)))
        subs[0](cur_stream(torch))
        us = per_launch_ms(torch, subs, max(reps, 2 * n_sets)) * 1000.0
        res["sublayer_k11_d5"] = rate(2 * 2.0 * Ch * Ch * 11 * T, 4 * T * Ch * 5, us, launches=2)
        for wt in ws.values():
            wt.close()
        out[f"{Ch}x{T}"] = res
        del bufs, Rs, x0
    # the upsamplers, leaky_relu(0.1) -> ConvTranspose1d -> crop -> + bias
    # (hift_vocoder.cpp:680-687), on the chain from 750 mel frames:
    # 512x750 -> 256x6000 -> 128x30000 -> 64x90000; algorithmic FLOPs
    # 2*C_in*C_out*K*T_in
    ups = {}
    for (Ci, Co, s, K, T) in ((512, 256, 8, 16, 750), (256, 128, 5, 11, 6000), (128, 64, 3, 7, 30000)):
        pad = (K - s) // 2
        T_out = (T - 1) * s + K - 2 * pad
        nbytes = 4 * (T * Ci + T_out * Co)
        n_sets = sets_for(nbytes)
        x0 = d(W.normal(W.seed_of(8, 1000 + Ci), (T, Ci)))
        bufs = [{"x": x0 if i == 0 else x0.clone(),
                 "y": torch.empty((T_out, Co), dtype=torch.float32, device="cuda")} for i in range(n_sets)]
        bias = d(W.normal(W.seed_of(8, 1001 + Ci), (Co,), 0.0, 0.1))
        wt = C.Conv1dWeights(d(W.normal(W.seed_of(8, 1002 + Ci), (Ci, Co, K), 0.0, 1.0 / np.sqrt(Ci * K / s))),
                             transpose_stride=s)
        rb = C.ctypes.byref(C.desc(bias))
        Rs = [{k: C.ctypes.byref(C.desc(v)) for k, v in b.items()} for b in bufs]
        fns = [lambda st, R=R: check_rc(C, L.cbx_conv_transpose1d(R["x"], wt.handle, pad, C.CONV_PRO_LEAKY_RELU,
                                                                   None, None, 0.1, rb, R["y"], st)) for R in Rs]
        fns[0](cur_stream(torch))
        us = per_launch_ms(torch, fns, max(reps, 2 * n_sets)) * 1000.0
        ups[f"{Ci}x{T}_to_{Co}x{T_out}"] = rate(2.0 * Ci * Co * K * T, nbytes, us, buffer_sets=n_sets)
        wt.close()
        del bufs, Rs, x0
    out["upsample"] = ups
    # the CFM decoder's causal_block1d conv: mul(x, mask) -> CausalConv1d K 3
    # (+ bias), cfm_decoder.cpp:89-120,139-142, on [2, C_in, 500] frames
    # (the CFG pair); algorithmic FLOPs 2*C_in*C_out*3*T*B
    cfm = {}
    for (Ci, Co, T, B) in ((256, 256, 500, 2), (512, 256, 500, 2)):
        nbytes = 4 * B * T * (Ci + Co)
        n_sets = sets_for(nbytes)
        x0 = d(W.normal(W.seed_of(8, 2000 + Ci), (B, T, Ci)))
        bufs = [{"x": x0 if i == 0 else x0.clone(), "y": torch.empty((B, T, Co), dtype=torch.float32, device="cuda")}
                for i in range(n_sets)]
        mask = torch.ones(T, dtype=torch.float32, device="cuda")
        bias = d(W.normal(W.seed_of(8, 2001 + Ci), (Co,), 0.0, 0.1))
        wt = C.Conv1dWeights(d(W.normal(W.seed_of(8, 2002 + Ci), (Co, Ci, 3), 0.0, 1.0 / np.sqrt(Ci * 3))))
        rm, rb = C.ctypes.byref(C.desc(mask)), C.ctypes.byref(C.desc(bias))
        Rs = [{k: C.ctypes.byref(C.desc(v)) for k, v in b.items()} for b in bufs]
        fns = [lambda st, R=R: check_rc(C, L.cbx_causal_conv1d(R["x"], wt.handle, rm, rb, R["y"], st)) for R in Rs]
        fns[0](cur_stream(torch))
        us = per_launch_ms(torch, fns, max(reps, 2 * n_sets)) * 1000.0
        cfm[f"{B}x{Ci}x{T}_to_{Co}"] = rate(2.0 * Ci * Co * 3 * T * B, nbytes, us, buffer_sets=n_sets)
        wt.close()
        del bufs, Rs, x0
    out["cfm_causal_conv"] = cfm
    return out


def bench_hift(C, W, torch, quick=False):
    """HiFT vocoder activations: Snake (channel innermost as the reference
    lays it out, and time innermost) and LeakyReLU(0.1) on every upsample
    stage shape; buffer sets rotate past the Infinity Cache.  x ~ N(0,1)
    from torch's seeded device generator (the tensors reach 123M elements)."""
    L = C.load()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(W.seed_of(4, 0))
    out = {}
    shapes = W.HIFT_SHAPES[-1:] if quick else W.HIFT_SHAPES
    for (B, Ch, T) in shapes:
        n = B * Ch * T
        a_np, ai_np = W.snake_alpha(Ch)
        a, ai = torch.from_numpy(a_np).cuda(), torch.from_numpy(ai_np).cuda()
        per = 8 * n
        n_sets = max(2, math.ceil(MALL_DEFEAT_BYTES / per))
        xs = [torch.empty((B, T, Ch), dtype=torch.float32, device="cuda").normal_(generator=gen) for _ in range(n_sets)]
        ys = [torch.empty_like(x) for x in xs]
        ra, rai = C.ctypes.byref(C.desc(a)), C.ctypes.byref(C.desc(ai))
        a_o, ai_o = a.view(Ch, 1), ai.view(Ch, 1)
        rao, raio = C.ctypes.byref(C.desc(a_o)), C.ctypes.byref(C.desc(ai_o))
        rx = [C.ctypes.byref(C.desc(x)) for x in xs]
        ry = [C.ctypes.byref(C.desc(y)) for y in ys]
        rxo = [C.ctypes.byref(C.desc(x.view(B, Ch, T))) for x in xs]
        ryo = [C.ctypes.byref(C.desc(y.view(B, Ch, T))) for y in ys]
        plans = {
            "snake_channel_inner": [(lambda i: lambda s: check_rc(C, L.cbx_snake(rx[i], ra, rai, ry[i], s)))(i)
                                    for i in range(n_sets)],
            "snake_time_inner": [(lambda i: lambda s: check_rc(C, L.cbx_snake(rxo[i], rao, raio, ryo[i], s)))(i)
                                 for i in range(n_sets)],
            "leaky_relu_0.1": [(lambda i: lambda s: check_rc(C, L.cbx_leaky_relu(rx[i], 0.1, ry[i], s)))(i)
                               for i in range(n_sets)],
        }
        key = f"{B}x{Ch}x{T}"
        out[key] = {"bytes": per + (8 * Ch), "buffer_sets": n_sets}
        reps = max(n_sets, min(200, int(2e10 / per)))
        for name, fns in plans.items():
            for f in fns:
                f(cur_stream(torch))
            ms = per_launch_ms(torch, fns, reps)
            nbytes = per + (8 * Ch if name.startswith("snake") else 0)
            out[key][name] = {"us": ms * 1000.0, "GBps": nbytes / (ms * 1e-3) / 1e9}
        del xs, ys
        torch.cuda.empty_cache()
    return out


def bench_copy_ceiling(C, torch, sizes, reps=400):
    """A plain f32 device copy (cbx_cpy: one read, one write, nothing else)
    of each byte count, over rotating buffers: the best rate a launch moving
    that many bytes reaches on this GPU, the practical ceiling of a kernel
    of the same size."""
    L = C.load()
    out = {}
    for name, nbytes in sizes.items():
        n = nbytes // 8
        n_sets = max(2, math.ceil(MALL_DEFEAT_BYTES / (2 * 4 * n)))
        xs = [torch.empty(n, dtype=torch.float32, device="cuda").uniform_() for _ in range(n_sets)]
        ys = [torch.empty_like(x) for x in xs]
        rx = [C.ctypes.byref(C.desc(x)) for x in xs]
        ry = [C.ctypes.byref(C.desc(y)) for y in ys]
        fns = [(lambda i: lambda s: check_rc(C, L.cbx_cpy(rx[i], ry[i], s)))(i) for i in range(n_sets)]
        for f in fns:
            f(cur_stream(torch))
        ms = per_launch_ms(torch, fns, reps)
        out[name] = {"bytes": 8 * n, "us": ms * 1000.0, "GBps": 8 * n / (ms * 1e-3) / 1e9}
        del xs, ys
    return out


TRAFFIC_FILE = os.path.join(ROOT, "profiles", "hbm_traffic_per_kernel_all_workloads.md")


def recorded_traffic(key):
    """HBM bytes per launch of a kernel as last measured with rocprofv3 --pmc
    FETCH_SIZE and WRITE_SIZE (copy-calibrated), or None."""
    try:
        with open(TRAFFIC_FILE) as f:
            for line in f:
                if line.startswith(f"traffic_bytes_per_launch {key}:"):
                    return int(float(line.split(":", 1)[1]))
    except OSError:
        pass
    return None


COPY_PROBE_ELEMS = 16 << 20   # the calibration copy: 64 MiB in, 64 MiB out


STATS_FILE = os.path.join(ROOT, "profiles", "prefill_chain_one_launch_kernel_stats.md")
ROOFLINE_KERNEL = "cbx::k_batch<516u>"


def recorded_kernel_avg_us(kernel):
    """A kernel's average duration (us) in the committed rocprofv3 kernel
    stats of the headline workload, or None."""
    try:
        with open(STATS_FILE) as f:
            for line in f:
                if line.startswith(f"| `{kernel}` |"):
                    return float(line.split("|")[3])
    except (OSError, ValueError, IndexError):
        pass
    return None


def traffic_groups(W):
    """The counter probe's launch groups in launch order: (label, algorithmic
    bytes per launch, launches).  Each group runs on its own buffer sets
    (one per launch; two for the 983 MB vocoder shape)."""
    nb, cb, bb, sb = W.prefill_bytes(), W.cfm_bytes(), W.t3_block_bytes(), W.serving_bytes()
    hift = {}
    for (B, Ch, T) in (W.HIFT_SHAPES[0], W.HIFT_SHAPES[-1]):
        hift[(B, Ch, T)] = 8 * B * Ch * T
    (s0, s1) = W.HIFT_SHAPES[0], W.HIFT_SHAPES[-1]
    return [
        ("copy_64MiB", 2 * 4 * COPY_PROBE_ELEMS, 4),
        ("copy_4KiB", 2 * 4096, 8),
        ("prefill_chain_one_launch", sum(nb.values()), 8),
        ("gelu_512x4096", nb["gelu"], 8),
        ("embed_layer_norm_512x1024", nb["embed_layer_norm"], 8),
        ("group_norm_mish_2x256x500", cb["group_norm_mish_256"], 8),
        ("group_norm_mish_2x512x500", cb["group_norm_mish_512"], 8),
        ("layer_norm_rope_2x500x512", cb["layer_norm_rope"], 8),
        ("residual_join_layer_norm_512x1024", bb["residual_ln2"], 8),
        ("bias_gelu_512x4096", bb["fc_bias_gelu"], 8),
        ("snake_1x256x6000", hift[s0] + 8 * s0[1], 8),
        ("leaky_relu_1x256x6000", hift[s0], 8),
        ("snake_16x64x120000", hift[s1] + 8 * s1[1], 2),
        ("leaky_relu_16x64x120000", hift[s1], 2),
        ("rms_norm_64x1024_f16", sb["rms_norm_mul"], 8),
        ("rope_64x16x64_f16", sb["rope_qk"] // 2, 8),
        ("swiglu_64x4096_f16", sb["swiglu"], 8),
        ("get_rows_q8_0_64x1024", sb["get_rows_q8_0"], 8),
        ("serving_step_one_launch", sum(sb.values()), 8),
        ("flow_step_one_launch", sum(cb.values()), 8),
        ("causal_conv1d_2x256x500", 4 * 2 * 500 * (256 + 256) + 2 * 256 * 256 * 3 + 4 * 256 + 4 * 500, 8),
    ]


def traffic_probe(C, W, torch):
    """The launches of the FETCH_SIZE / WRITE_SIZE counter runs: every buffer
    is made first, then the groups of traffic_groups() run in order, each
    kernel on its own buffer sets, with a device synchronisation between
    groups (so the profiler's dispatch order is the groups' order)."""
    L = C.load()
    d = dev_of(torch)
    s = cur_stream(torch)
    R = lambda t, ty=None: C.ctypes.byref(C.desc(t, ty))  # noqa: E731
    groups = {}
    x = torch.empty(COPY_PROBE_ELEMS, dtype=torch.float32, device="cuda").uniform_()
    ys = [torch.empty_like(x) for _ in range(4)]
    groups["copy_64MiB"] = [(lambda y: lambda: L.cbx_cpy(R(x), R(y), s))(y) for y in ys]
    small = [(torch.empty(1024, dtype=torch.float32, device="cuda").uniform_(),
              torch.empty(1024, dtype=torch.float32, device="cuda")) for _ in range(8)]
    groups["copy_4KiB"] = [(lambda a_, b_: lambda: L.cbx_cpy(R(a_), R(b_), s))(a_, b_) for a_, b_ in small]
    inp = W.prefill_inputs()
    pre = [PrefillSet(C, W, torch, inp) for _ in range(8)]
    groups["prefill_chain_one_launch"] = [(lambda st_: lambda: st_.step_one_launch(s))(st_) for st_ in pre]
    groups["gelu_512x4096"] = [(lambda st_: lambda: st_.gelu(s))(st_) for st_ in pre]
    groups["embed_layer_norm_512x1024"] = [(lambda st_: lambda: st_.embed_layer_norm(s))(st_) for st_ in pre]
    cfm = W.cfm_inputs()
    cache = C.RopeCache(W.HEAD_DIM, mode=2, n_ctx_orig=2048, n_pos=2048)
    ws = C.GroupNormWorkspace()
    cs = []
    for _ in range(8):
        t = {k: d(v) for k, v in cfm.items()}
        for k in ("x256", "x512", "xa"):
            t["y" + k[1:]] = torch.empty_like(t[k])
        cs.append({k: R(v) for k, v in t.items()} | {"_t": t})
    for key in ("256", "512"):
        groups[f"group_norm_mish_2x{key}x500"] = [
            (lambda r, key=key: lambda: L.cbx_group_norm_ws(r["x" + key], W.CFM_GROUPS, 1e-5, r["w" + key],
                                                            r["b" + key], C.MISH, r["y" + key], ws.handle, s))(r)
            for r in cs]
    groups["layer_norm_rope_2x500x512"] = [
        (lambda r: lambda: L.cbx_layer_norm_rope(r["xa"], r["wa"], r["ba"], 1e-5, W.HEAD_DIM, r["pos"], cache.handle,
                                                 r["ya"], s))(r) for r in cs]
    blk = W.t3_block_inputs()
    N, D, F = W.N_PREFILL, W.D_MODEL, W.D_FF
    bs = []
    for _ in range(8):
        t = {k: d(blk[k]) for k in ("attn_mm", "h", "out_b", "ln2_w", "ln2_b", "fc_mm", "fc_b")}
        t["res"], t["ln2"] = torch.empty((N, D), device="cuda"), torch.empty((N, D), device="cuda")
        t["gelu"] = torch.empty((N, F), device="cuda")
        bs.append({k: R(v) for k, v in t.items()} | {"_t": t})
    groups["residual_join_layer_norm_512x1024"] = [
        (lambda r: lambda: L.cbx_add_layer_norm(r["attn_mm"], r["out_b"], r["h"], r["ln2_w"], r["ln2_b"], 1e-5, -1,
                                                r["res"], r["ln2"], s))(r) for r in bs]
    groups["bias_gelu_512x4096"] = [(lambda r: lambda: L.cbx_bias_act(C.GELU, r["fc_mm"], r["fc_b"], r["gelu"], s))(r)
                                    for r in bs]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(W.seed_of(4, 0))
    hb = []
    for (B, Ch, T), n_sets in ((W.HIFT_SHAPES[0], 8), (W.HIFT_SHAPES[-1], 2)):
        a, ai = (d(v) for v in W.snake_alpha(Ch))
        sets_ = []
        for _ in range(n_sets):
            xx = torch.empty((B, T, Ch), dtype=torch.float32, device="cuda").normal_(generator=gen)
            sets_.append((xx, torch.empty_like(xx)))
        hb.append((a, ai, sets_))
        tag = f"{B}x{Ch}x{T}"
        groups[f"snake_{tag}"] = [(lambda xx, yy, a=a, ai=ai: lambda: L.cbx_snake(R(xx), R(a), R(ai), R(yy), s))(xx, yy)
                                  for xx, yy in sets_]
        groups[f"leaky_relu_{tag}"] = [(lambda xx, yy: lambda: L.cbx_leaky_relu(R(xx), 0.1, R(yy), s))(xx, yy)
                                       for xx, yy in sets_]
    sv_base = {k: d(v) for k, v in W.serving_inputs().items()}
    sv = []
    for _ in range(8):
        t = {k: v.clone() for k, v in sv_base.items()}
        t["y"], t["qo"], t["ko"] = torch.empty_like(t["x"]), torch.empty_like(t["q"]), torch.empty_like(t["k"])
        t["h"] = torch.empty_like(t["gate"])
        t["emb"] = torch.empty((W.N_STREAMS, W.D_MODEL), dtype=torch.float32, device="cuda")
        r = {k: R(v, C.Q8_0 if k == "tab" else None) for k, v in t.items()}
        one = C.OpBatch([C.Op(C.OP_RMS_NORM, [t["x"], t["g"]], [t["y"]], eps=1e-5),
                         C.Op(C.OP_ROPE, [t["q"], t["pos"]], [t["qo"]], rope=cache),
                         C.Op(C.OP_ROPE, [t["k"], t["pos"]], [t["ko"]], rope=cache),
                         C.Op(C.OP_SWIGLU, [t["gate"], t["up"]], [t["h"]]),
                         C.Op(C.OP_GET_ROWS, [t["tab"], t["ids"]], [t["emb"]], q8=[0])])
        sv.append((t, r, one))
    groups["rms_norm_64x1024_f16"] = [(lambda r: lambda: L.cbx_rms_norm_mul(r["x"], r["g"], 1e-5, r["y"], s))(r)
                                      for _, r, _ in sv]
    groups["rope_64x16x64_f16"] = [(lambda r: lambda: L.cbx_rope_ext(r["q"], r["pos"], cache.handle, r["qo"], s))(r)
                                   for _, r, _ in sv]
    groups["swiglu_64x4096_f16"] = [(lambda r: lambda: L.cbx_swiglu(r["gate"], r["up"], r["h"], s))(r) for _, r, _ in sv]
    groups["get_rows_q8_0_64x1024"] = [(lambda r: lambda: L.cbx_get_rows(r["tab"], r["ids"], r["emb"], s))(r)
                                       for _, r, _ in sv]
    groups["serving_step_one_launch"] = [(lambda one: lambda: L.cbx_run_ops(one.arr, one.n, s))(one) for _, _, one in sv]
    flow = []
    for r in cs:
        t = r["_t"]
        flow.append(C.OpBatch([
            C.Op(C.OP_GROUP_NORM, [t["x256"], t["w256"], t["b256"]], [t["y256"]], act=C.MISH, eps=1e-5,
                 iparam=W.CFM_GROUPS),
            C.Op(C.OP_GROUP_NORM, [t["x512"], t["w512"], t["b512"]], [t["y512"]], act=C.MISH, eps=1e-5,
                 iparam=W.CFM_GROUPS),
            C.Op(C.OP_LAYER_NORM_ROPE, [t["xa"], t["wa"], t["ba"], t["pos"]], [t["ya"]], eps=1e-5, rope=cache,
                 iparam=W.HEAD_DIM)]))
    groups["flow_step_one_launch"] = [(lambda one: lambda: L.cbx_run_ops(one.arr, one.n, s))(one) for one in flow]
    cc = []
    wt = C.Conv1dWeights(d(W.normal(W.seed_of(8, 2002 + 256), (256, 256, 3), 0.0, 1.0 / np.sqrt(256 * 3))))
    mask = torch.ones(500, dtype=torch.float32, device="cuda")
    bias = d(W.normal(W.seed_of(8, 2001 + 256), (256,), 0.0, 0.1))
    for _ in range(8):
        xx = d(W.normal(W.seed_of(8, 2000 + 256), (2, 500, 256)))
        cc.append((xx, torch.empty_like(xx)))
    groups["causal_conv1d_2x256x500"] = [
        (lambda xx, yy: lambda: L.cbx_causal_conv1d(R(xx), wt.handle, R(mask), R(bias), R(yy), s))(xx, yy)
        for xx, yy in cc]
    torch.cuda.synchronize()
    for label, nbytes, n in traffic_groups(W):
        fns = groups[label]
        assert len(fns) == n, label
        for fn in fns:
            check_rc(C, fn())
        torch.cuda.synchronize()
        log(f"traffic probe: {label} x{n}")
    cache.close()
    ws.close()
    wt.close()
    print(json.dumps({"groups": [[lb, nbytes, n] for lb, nbytes, n in traffic_groups(W)]}), flush=True)


def _pmc_dispatches(d):
    """(kernel name, {counter: value}) of every dispatch of ours in a
    rocprofv3 --pmc csv run, in dispatch order."""
    import csv
    import glob
    f = sorted(glob.glob(os.path.join(d, "**", "*counter_collection.csv"), recursive=True))[0]
    by = {}
    for r in csv.DictReader(open(f)):
        # cbx_init's XCD probe runs once before any probe group
        if "cbx::" not in r["Kernel_Name"] or "k_xcc_probe" in r["Kernel_Name"]:
            continue
        k = int(r["Dispatch_Id"])
        by.setdefault(k, (r["Kernel_Name"], {}))[1][r["Counter_Name"]] = float(r["Counter_Value"])
    return [by[k] for k in sorted(by)]


def _pmc_rows(d):
    """(kernel name, counter value) of every dispatch of a one-counter
    rocprofv3 --pmc csv run, in dispatch order."""
    return [(k, next(iter(c.values()))) for k, c in _pmc_dispatches(d)]


def _group_medians(W, d):
    """Per traffic_groups() entry: (label, algorithmic bytes, launches,
    kernel, {counter: median over its launches})."""
    rows = _pmc_dispatches(d)
    groups = traffic_groups(W)
    total = sum(n for _, _, n in groups)
    if len(rows) != total:
        raise SystemExit(f"counter summary: {len(rows)} dispatches of ours in {d}, {total} expected")
    out, i = [], 0
    for label, nbytes, n in groups:
        names = sorted(rows[i][1])
        med = {c: sorted(r[1][c] for r in rows[i:i + n])[n // 2] for c in names}
        out.append((label, nbytes, n, short_kernel(rows[i][0]), med))
        i += n
    return out


def counters_summary(W, title, command, *dirs):
    """Markdown of --pmc runs over --traffic-probe (one directory a pass):
    every group's median counter values, plus, when the read-request
    counters are there, the bytes they imply by request size and, when the
    occupancy counters are there, waves per active CU."""
    per = None
    for d in dirs:
        g = _group_medians(W, d)
        per = g if per is None else [(a[0], a[1], a[2], a[3], {**a[4], **b[4]}) for a, b in zip(per, g)]
    names = sorted({c for p in per for c in p[4]})
    out = [f"# {title}", "", "Command (one MI355X):", "", "```", f"cd /tmp && export TMPDIR=/tmp && cd {ROOT}",
           command, "```", "", "Median over each group's launches (one launch per buffer set; groups as "
           "`traffic_groups()` in bench.py).", "",
           "| workload | kernel | " + " | ".join(names) + " |", "|---|---|" + "---|" * len(names)]
    for label, nbytes, n, kern, med in per:
        out.append(f"| {label} | `{kern}` | " + " | ".join(f"{med.get(c, float('nan')):.4g}" for c in names) + " |")
    if {"TCC_EA0_RDREQ_sum", "TCC_EA0_RDREQ_32B_sum", "TCC_BUBBLE_sum"} <= set(names):
        c = per[0][4]
        per_req = 4 * COPY_PROBE_ELEMS / c["TCC_EA0_RDREQ_sum"]
        out += ["", f"The 64 MiB copy reads {4 * COPY_PROBE_ELEMS} bytes in {c['TCC_EA0_RDREQ_sum']:.0f} L2-to-memory "
                f"read requests: {per_req:.2f} bytes a request, one 128-byte line each, while TCC_BUBBLE (the "
                "128-byte request count) and TCC_EA0_RDREQ_32B read 0 for every kernel.  FETCH_SIZE's formula "
                "(128 x TCC_BUBBLE + 64 x the other requests + 32 x the 32-byte ones) therefore counts each "
                "128-byte line as 64 bytes: the factor 2 that scales FETCH_SIZE.  Per kernel, the requests at "
                "128 bytes against the lines its algorithmic reads span (inputs once); the requests beyond those "
                "lines are what each launch fetches besides its data (kernel code and arguments into each XCD's "
                "L2, tables), a fixed few hundred a launch that shows only in kernels reading under a megabyte:",
                "", "| workload | read requests | bytes at 128 B a request | algorithmic read bytes | ratio | "
                "requests beyond the data's lines |", "|---|---|---|---|---|---|"]
        for label, nbytes, n, kern, med in per:
            r = med["TCC_EA0_RDREQ_sum"]
            rd = read_bytes_of(W, label, nbytes)
            lines = -(-rd // 128)
            out.append(f"| {label} | {r:.0f} | {128 * r:.0f} | {rd} | {128 * r / rd if rd else float('nan'):.3f} | "
                       f"{r - lines:.0f} |")
    if "MeanOccupancyPerActiveCU" in names:
        out += ["", "MeanOccupancyPerActiveCU is the average number of resident waves on a CU while it is busy (a "
                "CU holds at most 32: 8 per SIMD); OccupancyPercent the same over the whole launch and every CU; "
                "SQ_WAVES the waves the launch ran."]
    if "VALUUtilization" in names:
        out += ["", "VALUUtilization: the share of lanes active in the vector ALU instructions issued; VALUBusy: the "
                "share of the launch's time the vector ALUs issued (per CU)."]
    return "\n".join(out) + "\n"


def read_bytes_of(W, label, nbytes):
    """The algorithmic bytes a probe group's launch reads (inputs once)."""
    writes = {"copy_64MiB": 4 * COPY_PROBE_ELEMS, "copy_4KiB": 4096}
    sb, cb = W.serving_bytes(), W.cfm_bytes()
    if label in writes:
        return nbytes - writes[label]
    # outputs: f32 rows written once; the rest of the bytes are reads
    out = {"prefill_chain_one_launch": 2 * 512 * 1024 * 4 + 512 * 4096 * 4,
           "gelu_512x4096": 512 * 4096 * 4, "embed_layer_norm_512x1024": 2 * 512 * 1024 * 4,
           "group_norm_mish_2x256x500": 2 * 256 * 500 * 4, "group_norm_mish_2x512x500": 2 * 512 * 500 * 4,
           "layer_norm_rope_2x500x512": 2 * 500 * 512 * 4, "residual_join_layer_norm_512x1024": 2 * 512 * 1024 * 4,
           "bias_gelu_512x4096": 512 * 4096 * 4, "snake_1x256x6000": 256 * 6000 * 4,
           "leaky_relu_1x256x6000": 256 * 6000 * 4, "snake_16x64x120000": 16 * 64 * 120000 * 4,
           "leaky_relu_16x64x120000": 16 * 64 * 120000 * 4, "rms_norm_64x1024_f16": 64 * 1024 * 2,
           "rope_64x16x64_f16": 64 * 16 * 64 * 2, "swiglu_64x4096_f16": 64 * 4096 * 2,
           "get_rows_q8_0_64x1024": 64 * 1024 * 4,
           "serving_step_one_launch": 64 * 1024 * 2 + 2 * 64 * 16 * 64 * 2 + 64 * 4096 * 2 + 64 * 1024 * 4,
           "flow_step_one_launch": 2 * 256 * 500 * 4 + 2 * 512 * 500 * 4 + 2 * 500 * 512 * 4,
           "causal_conv1d_2x256x500": 2 * 500 * 256 * 4}
    return nbytes - out[label] if label in out else 0


def short_kernel(name):
    import re
    n = re.sub(r"\(anonymous namespace\)::", "", name)
    n = re.sub(r"^void ", "", n)
    return re.sub(r"\((cbx::|float const|char const|unsigned|cbx|long).*$", "", n)


def traffic_summary(W, fetch_dir, write_dir):
    """Markdown of two counter runs over --traffic-probe: each group's
    dispatches (our kernels, in dispatch order) matched to traffic_groups(),
    FETCH_SIZE and WRITE_SIZE scaled by what they read for the copy of known
    size."""
    F, Wr = _pmc_rows(fetch_dir), _pmc_rows(write_dir)
    groups = traffic_groups(W)
    total = sum(n for _, _, n in groups)
    if len(F) != total or len(Wr) != total:
        raise SystemExit(f"traffic summary: {len(F)} / {len(Wr)} dispatches of ours, {total} expected")
    per, i = [], 0
    for label, nbytes, n in groups:
        fs = sorted(v for _, v in F[i:i + n])
        ws_ = sorted(v for _, v in Wr[i:i + n])
        per.append((label, nbytes, n, short_kernel(F[i][0]), fs[len(fs) // 2], ws_[len(ws_) // 2]))
        i += n
    copy_kib = 4 * COPY_PROBE_ELEMS / 1024
    f_scale, w_scale = copy_kib / per[0][4], copy_kib / per[0][5]
    out = ["# HBM traffic per launch of every configuration's kernels (FETCH_SIZE, WRITE_SIZE)", "",
           "Two `rocprofv3 --pmc` passes on one MI355X over the same probe (a 64 MiB f32 copy of known size, then",
           "each kernel's launches on their own buffer sets; the groups are `traffic_groups()` in bench.py):", "",
           "```", f"cd /tmp && export TMPDIR=/tmp && cd {ROOT}",
           f"timeout -s KILL 120 rocprofv3 --pmc FETCH_SIZE --output-format csv -d {fetch_dir} -o run -- "
           "python -u bench.py --traffic-probe",
           f"timeout -s KILL 120 rocprofv3 --pmc WRITE_SIZE --output-format csv -d {write_dir} -o run -- "
           "python -u bench.py --traffic-probe",
           f"python bench.py --traffic-summary {fetch_dir} {write_dir}", "```", "",
           f"Calibration: the copy moves {copy_kib:.0f} KiB each way; FETCH_SIZE reads {per[0][4]:.1f} KiB for it "
           f"and WRITE_SIZE {per[0][5]:.1f}, so reads are scaled by {f_scale:.4f} and writes by {w_scale:.4f}.", "",
           "| workload | kernel | launches | FETCH_SIZE KiB | WRITE_SIZE KiB | algorithmic bytes | traffic bytes | ratio |",
           "|---|---|---|---|---|---|---|---|"]
    tail = []
    for label, nbytes, n, kern, fv, wv in per[1:]:
        traffic = (fv * f_scale + wv * w_scale) * 1024
        out.append(f"| {label} | `{kern}` | {n} | {fv:.1f} | {wv:.1f} | {nbytes} | {traffic:.0f} | "
                   f"{traffic / nbytes:.3f} |")
        tail.append(f"traffic_bytes_per_launch {label}: {traffic:.0f}")
    return "\n".join(out + [""] + tail) + "\n"


def stats_summary(stats_dir, title, command):
    """Markdown of a rocprofv3 --kernel-trace --stats run: our kernels'
    calls and durations."""
    import csv
    import glob
    f = sorted(glob.glob(os.path.join(stats_dir, "**", "*kernel_stats.csv"), recursive=True))[0]
    rows = [r for r in csv.DictReader(open(f)) if "cbx::" in r["Name"]]
    rows.sort(key=lambda r: -float(r["TotalDurationNs"]))
    out = [f"# {title}", "", "Command (one MI355X):", "", "```", f"cd /tmp && export TMPDIR=/tmp && cd {ROOT}",
           command, "```", "", "Kernels of libcbxops (rocprofv3 kernel stats; durations in microseconds):", "",
           "| kernel | calls | average | min | max |", "|---|---|---|---|---|"]
    for r in rows:
        out.append(f"| `{short_kernel(r['Name'])}` | {r['Calls']} | {float(r['AverageNs']) / 1e3:.3f} | "
                   f"{float(r['MinNs']) / 1e3:.3f} | {float(r['MaxNs']) / 1e3:.3f} |")
    return "\n".join(out) + "\n"


def cpu_baseline(W, seconds):
    """The oracle runs the same prefill chain on the host cores."""
    from oracle import oracle as O

    inp = W.prefill_inputs()
    per_step = sum(W.prefill_bytes(False).values())
    nth = max(1, min(16, os.cpu_count() or 1))
    reps = 0
    t0 = time.perf_counter()
    while True:
        h = O.get_rows_add(inp["table"], inp["ids"], inp["pos_table"], inp["pos_ids"], nth=nth)
        O.layer_norm(h, inp["ln_w"], inp["ln_b"], 1e-5, nth=nth)
        O.unary(O.GELU, inp["ffn"], nth=nth)
        reps += 1
        el = time.perf_counter() - t0
        if el >= seconds or reps >= 100000:
            break
    details = cpu_other_workloads(W, O, nth, max(1.0, seconds / 5.0))
    model = ""
    try:
        with open("/proc/cpuinfo") as f:
            model = next((ln.split(":", 1)[1].strip() for ln in f if ln.startswith("model name")), "")
    except OSError:
        pass
    return {"value": per_step * reps / el / 1e9, "unit": "GB/s", "cores": nth, "kind": "port",
            "sample": f"{reps} steps of the T3 prefill op chain (gather+pos f32, LayerNorm, GELU), "
                      f"{el:.1f} s, OpenMP row split as ggml-cpu",
            "nproc": os.cpu_count(), "cpu_model": model, "details": details}


def cpu_node_list(C, e):
    """A node-list builder's nodes as oracle.run_node_list takes them, the
    tensors' shapes, and seeded leaf values (normal f32; int32 leaves, the
    token ids and positions, 0, 1, 2, ...)."""
    import torch

    names = {C.GOP_VIEW: "view", C.GOP_GET_ROWS: "get_rows", C.GOP_ADD: "add", C.GOP_MUL: "mul",
             C.GOP_SCALE: "scale", C.GOP_NORM: "norm", C.GOP_SOFT_MAX: "soft_max", C.GOP_UNARY: "unary",
             C.GOP_LEAKY_RELU: "leaky_relu", C.GOP_ROPE: "rope"}
    nodes = [(names[n.op], n.dst, n.src[0], n.src[1], n.iparam, n.fparam) for n in e.graph.nodes]
    made = {n.dst for n in e.graph.nodes}
    n_t = len(e.graph._descs)
    shapes = {i: tuple(e.b.at(i).shape) for i in range(n_t)}
    rng = np.random.default_rng(7)
    leaves = {}
    for i in range(n_t):
        if i in made:
            continue
        if e.b.at(i).dtype == torch.int32:
            leaves[i] = (np.arange(int(np.prod(shapes[i]))) % 1000).astype(np.int32).reshape(shapes[i])
        else:
            leaves[i] = rng.standard_normal(shapes[i]).astype(np.float32)
    return nodes, shapes, leaves


def _timed(fn, seconds):
    reps, t0 = 0, time.perf_counter()
    while True:
        fn()
        reps += 1
        el = time.perf_counter() - t0
        if el >= seconds or reps >= 100000:
            return reps, el


def cpu_other_workloads(W, O, nth, seconds):
    """The oracle on the other workloads' shapes (same inputs as the GPU
    legs), a bounded sample each: decode step chain (us per step), the
    64-stream f16 step, a CFM flow step, a T3 block's element-wise nodes,
    one T3 decode token's element-wise nodes (24 blocks at N_new = 1, one
    thread: every op is one row), two HiFT stages' activations, a ResBlock
    conv and an upsampler."""
    out = {}
    steps = [W.decode_inputs(t) for t in range(W.DECODE_STEPS)]

    def decode():
        for d in steps:
            O.rms_norm_mul(d["x"], d["g"], 1e-5, nth=nth)
            O.rope_ext(d["q"], d["pos"], W.HEAD_DIM, mode=2, nth=nth)
            O.rope_ext(d["k"], d["pos"], W.HEAD_DIM, mode=2, nth=nth)
            O.swiglu(d["gate"], d["up"], nth=nth)
    reps, el = _timed(decode, seconds)
    out["t3_decode_us_per_step"] = el / (reps * W.DECODE_STEPS) * 1e6

    sv = W.serving_inputs()

    def serving():
        O.rms_norm_mul(sv["x"], sv["g"], 1e-5, nth=nth)
        O.rope_ext(sv["q"], sv["pos"], W.HEAD_DIM, mode=2, nth=nth)
        O.rope_ext(sv["k"], sv["pos"], W.HEAD_DIM, mode=2, nth=nth)
        O.swiglu(sv["gate"], sv["up"], nth=nth)
        O.get_rows(sv["tab"], sv["ids"], q8_0=True, nth=nth)
    reps, el = _timed(serving, seconds)
    out["serving_64_streams_f16_GBps"] = sum(W.serving_bytes().values()) * reps / el / 1e9

    cf = W.cfm_inputs()

    def flow():
        O.group_norm_affine(cf["x256"], W.CFM_GROUPS, 1e-5, cf["w256"], cf["b256"], True, nth=nth)
        O.group_norm_affine(cf["x512"], W.CFM_GROUPS, 1e-5, cf["w512"], cf["b512"], True, nth=nth)
        ln = O.layer_norm(cf["xa"], cf["wa"], cf["ba"], 1e-5, nth=nth)
        O.rope_ext(ln.reshape(2, W.CFM_T, W.CFM_HEADS, W.HEAD_DIM), cf["pos"], W.HEAD_DIM, mode=2, nth=nth)
    reps, el = _timed(flow, seconds)
    out["cfm_flow_step_GBps"] = sum(W.cfm_bytes().values()) * reps / el / 1e9

    blk = W.t3_block_inputs()

    def t3_block():
        res = O.add(O.add(blk["attn_mm"], blk["out_b"], nth=nth), blk["h"], nth=nth)
        O.layer_norm(res, blk["ln2_w"], blk["ln2_b"], 1e-5, nth=nth)
        O.unary(O.GELU, O.add(blk["fc_mm"], blk["fc_b"], nth=nth), nth=nth)
        h2 = O.add(O.add(blk["proj_mm"], blk["proj_b"], nth=nth), res, nth=nth)
        O.layer_norm(h2, blk["ln1_w"], blk["ln1_b"], 1e-5, nth=nth)
    reps, el = _timed(t3_block, seconds)
    bb = W.t3_block_bytes()
    out["t3_block_elementwise_GBps"] = (bb["residual_ln2"] + bb["fc_bias_gelu"] + bb["residual_next_ln1"]) * reps / el / 1e9

    tok = O.T3TokenStep(W.t3_token_inputs(), 255)
    reps, el = _timed(lambda: tok.run(17, 255), seconds)
    out["t3_token_elementwise_us_per_token_1thread"] = el / reps * 1e6

    # the encoder calls' node lists run node by node on the oracle, as
    # ggml-cpu runs a graph (same lists and sizes as the GPU legs)
    from chatterbox_amdvulkan_amd import cbxops as C
    from chatterbox_amdvulkan_amd.flow_encoder import FlowEncoderCall
    from chatterbox_amdvulkan_amd.s3_encoder import HEAD_DIM, ROPE_BASE, ROPE_MAX, S3EncoderCall

    rope = dict(n_dims=HEAD_DIM, mode=2, n_ctx_orig=ROPE_MAX, freq_base=ROPE_BASE)
    for name, e in (("flow_encoder", FlowEncoderCall(250, device=False)), ("s3_encoder", S3EncoderCall(1000, device=False))):
        nodes, shapes, leaves = cpu_node_list(C, e)
        reps, el = _timed(lambda: O.run_node_list(nodes, shapes, dict(leaves), rope=rope, nth=nth), seconds)
        out[f"{name}_call_us"] = el / reps * 1e6

    for (B, Ch, T) in W.HIFT_SHAPES[:3:2]:
        x = W.normal(W.seed_of(4, 2), (B, T, Ch))
        a, ai = W.snake_alpha(Ch)
        reps, el = _timed(lambda: O.snake(x, a, ai, nth=nth), seconds)
        out[f"hift_snake_{B}x{Ch}x{T}_GBps"] = (8 * x.size + 8 * Ch) * reps / el / 1e9
        reps, el = _timed(lambda: O.leaky_relu(x, 0.1, nth=nth), seconds)
        out[f"hift_leaky_{B}x{Ch}x{T}_GBps"] = 8 * x.size * reps / el / 1e9
    xc = W.normal(W.seed_of(8, 64), (2000, 64))
    wc = W.normal(W.seed_of(8, 75), (64, 64, 11), 0.0, 0.04)
    ac, aic = W.snake_alpha(64, 3)
    reps, el = _timed(lambda: O.conv1d(xc, wc, 1, 25, 5, O.CONV_PRO_SNAKE, ac, aic, nth=nth), seconds)
    out["hift_conv_64x2000_k11_d5_GFLOPs"] = 2.0 * 64 * 64 * 11 * 2000 * reps / el / 1e9
    xu = W.normal(W.seed_of(8, 1100), (500, 128))
    wu = W.normal(W.seed_of(8, 1101), (128, 64, 7), 0.0, 0.05)
    reps, el = _timed(lambda: O.conv_transpose1d(xu, wu, 3, 2, O.CONV_PRO_LEAKY, slope=0.1, nth=nth), seconds)
    out["hift_upsample_128x500_s3_k7_GFLOPs"] = 2.0 * 128 * 64 * 7 * 500 * reps / el / 1e9
    return out


def main():
    a = parse()
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if a.gpus != 1 or world != 1:
        print("bench.py measures one GPU: this op path has no cross-GPU exchange and runs on one "
              "device; --gpus above 1 is not supported.", file=sys.stderr)
        return 2
    from chatterbox_amdvulkan_amd import workloads as W

    if a.traffic_summary:
        print(traffic_summary(W, *a.traffic_summary), end="")
        return 0
    if a.stats_summary:
        print(stats_summary(*a.stats_summary), end="")
        return 0
    if a.counters_summary:
        print(counters_summary(W, *a.counters_summary), end="")
        return 0
    import torch

    from chatterbox_amdvulkan_amd import cbxops as C

    torch.cuda.set_device(0)
    C.init(0)
    if a.traffic_probe:
        traffic_probe(C, W, torch)
        return 0
    if a.hift_conv:
        print(json.dumps({"hift_resblock_conv": bench_hift_conv(C, W, torch)}), flush=True)
        return 0
    if a.only:
        nb = W.prefill_bytes()
        fn = {"decode": lambda: bench_decode(C, W, torch), "serving": lambda: bench_serving(C, W, torch),
              "cfm": lambda: bench_cfm(C, W, torch), "hift": lambda: bench_hift(C, W, torch),
              "softmax": lambda: bench_softmax(C, W, torch), "t3_block": lambda: bench_t3_block(C, W, torch),
              "t3_token": lambda: bench_t3_token(C, W, torch),
              "cfm_estimator": lambda: bench_cfm_estimator(C, torch),
              "hift_decode": lambda: bench_hift_decode(C, torch),
              "s3_encoder": lambda: bench_s3_encoder(C, torch),
              "flow_encoder": lambda: bench_flow_encoder(C, torch),
              "hift_conv": lambda: bench_hift_conv(C, W, torch),
              "copy": lambda: bench_copy_ceiling(C, torch, {"gelu_bytes": nb["gelu"],
                                                            "embed_layer_norm_bytes": nb["embed_layer_norm"],
                                                            "chain_bytes": sum(nb.values()),
                                                            "group_norm_256_bytes": W.cfm_bytes()["group_norm_mish_256"],
                                                            "group_norm_512_bytes": W.cfm_bytes()["group_norm_mish_512"]})}
        print(json.dumps({a.only: fn[a.only]()}), flush=True)
        return 0
    # the chain's two ops (embedding + LayerNorm, GELU) are independent here:
    # the headline runs them as one launch (cbx_run_ops)
    res = bench_prefill(C, W, torch, a.steps, a.warmup, one_launch=True)

    def gbps(r):
        return r["bytes_per_step"] / (r["ms_per_step"] * 1e-3) / 1e9

    details = {"prefill_f32_one_launch": dict(res, GBps=gbps(res))}
    r2 = bench_prefill(C, W, torch, a.steps, a.warmup)
    details["prefill_f32_fused_two_launches"] = dict(r2, GBps=gbps(r2))
    if not a.quick:
        ru = bench_prefill(C, W, torch, max(200, a.steps // 4), 20, fused=False)
        details["prefill_f32_unfused"] = dict(ru, GBps=gbps(ru))
        r16 = bench_prefill(C, W, torch, max(200, a.steps // 4), 20, f16_table=True)
        details["prefill_f16_table_fused"] = dict(r16, GBps=gbps(r16))
        rr = bench_prefill(C, W, torch, max(200, a.steps // 4), 20, resident=True)
        details["prefill_f32_fused_cache_resident"] = dict(rr, GBps=gbps(rr))
        nb = W.prefill_bytes()
        cb = W.cfm_bytes()
        details["copy_ceiling"] = bench_copy_ceiling(C, torch, {"gelu_bytes": nb["gelu"],
                                                                "embed_layer_norm_bytes": nb["embed_layer_norm"],
                                                                "chain_bytes": sum(nb.values()),
                                                                "group_norm_256_bytes": cb["group_norm_mish_256"],
                                                                "group_norm_512_bytes": cb["group_norm_mish_512"]})
        log("decode")
        details["t3_decode"] = bench_decode(C, W, torch)
        log("serving")
        details["serving_64_streams_f16"] = bench_serving(C, W, torch)
        log("cfm")
        details["cfm_flow_step"] = bench_cfm(C, W, torch)
        log("hift")
        details["hift_activations"] = bench_hift(C, W, torch)
        log("softmax")
        details["attention_softmax"] = bench_softmax(C, W, torch)
        log("t3 block")
        details["t3_block_elementwise"] = bench_t3_block(C, W, torch)
        log("t3 token")
        details["t3_token_elementwise"] = bench_t3_token(C, W, torch)
        log("cfm estimator")
        details["cfm_estimator_elementwise"] = bench_cfm_estimator(C, torch)
        log("hift decode")
        details["hift_decode"] = bench_hift_decode(C, torch)
        log("s3 encoder")
        details["s3_encoder_elementwise"] = bench_s3_encoder(C, torch)
        log("flow encoder")
        details["flow_encoder_elementwise"] = bench_flow_encoder(C, torch)
        log("hift conv")
        details["hift_resblock_conv"] = bench_hift_conv(C, W, torch)
    k_ms = res["kernel_ms"]["run_ops"]
    k_bytes = res["bytes_per_step"]
    rp_us = recorded_kernel_avg_us(ROOFLINE_KERNEL)
    achieved_live = k_bytes / (k_ms * 1e-3) / 1e9
    # the roofline figure of record follows from the committed rocprof
    # summary (its average traced duration of this kernel); the live
    # back-to-back figure is reported beside it
    achieved = k_bytes / (rp_us * 1e-6) / 1e9 if rp_us else achieved_live
    value = res["bytes_per_step"] / (res["ms_per_step"] * 1e-3) / 1e9
    out = {
        "metric": "fused-op HBM GB/s (% of peak) + T3 per-token norm/rope/act µs, 1 GPU",
        "value": round(value, 2),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": a.steps,
        "warmup": a.warmup,
        "ms_per_step": res["ms_per_step"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": "t3_prefill_op_chain",
                   "embed_layer_norm": "512 ids of [8194,1024] f32 + pos rows 0..511, then LayerNorm eps 1e-5 "
                                       "affine, writing h and LN(h)",
                   "gelu": "[512,4096] tanh (fp16-table semantics)",
                   "launches": "one (cbx_run_ops: both ops, independent inputs)",
                   "hbm_pct_of_peak": round(100.0 * value / PEAK_HBM_GBS, 2),
                   "buffer_sets": res["n_sets"]},
        "roofline": {"bound": "hbm", "kernel": "k_batch: embedding+LayerNorm [512,1024] and GELU [512,4096]",
                     "achieved": round(achieved, 2),
                     "peak": PEAK_HBM_GBS, "unit": "GB/s", "frac": round(achieved / PEAK_HBM_GBS, 4),
                     "traffic": recorded_traffic("prefill_chain_one_launch"),
                     "traffic_source": os.path.relpath(TRAFFIC_FILE, ROOT),
                     "algorithmic_bytes": k_bytes,
                     "achieved_from": "rocprof_avg_us" if rp_us else "live",
                     "rocprof_avg_us": rp_us,
                     "rocprof_source": os.path.relpath(STATS_FILE, ROOT),
                     "launch_ms_live": k_ms, "achieved_live": round(achieved_live, 2),
                     "frac_live": round(achieved_live / PEAK_HBM_GBS, 4)},
    }
    if "t3_decode" in details:
        dd = details["t3_decode"]
        out["t3_decode_us_per_step_chain"] = {k: round(dd[k]["us_per_step"], 3)
                                              for k in ("per_op_4_launches", "qk_merged_3_launches", "one_launch")}
    if "t3_token_elementwise" in details:
        tt = details["t3_token_elementwise"]
        out["t3_per_token_us"] = {"reference_sequence": "t3.cpp:446-546 at N_new = 1, 24 blocks, "
                                                        f"{tt['launches']} launches, n_past {tt['n_past']}",
                                  "exec_replay": round(tt["exec_replay_us_per_token"], 2),
                                  "decode_loop_with_update": round(tt["decode_loop_us_per_token"], 2)}
    if "cfm_estimator_elementwise" in details:
        ce = details["cfm_estimator_elementwise"]
        out["cfm_estimator_us_per_call"] = {"reference_sequence": ce["reference_sequence"] +
                                            f", {ce['launches']} launches",
                                            "exec_replay": round(ce["exec_replay_us_per_call"], 2)}
    if "s3_encoder_elementwise" in details:
        se = details["s3_encoder_elementwise"]
        out["s3_encoder_us_per_call"] = {"reference_sequence": se["reference_sequence"] +
                                         f", {se['launches']} launches",
                                         "exec_replay": round(se["exec_replay_us_per_call"], 2)}
    if "flow_encoder_elementwise" in details:
        fe = details["flow_encoder_elementwise"]
        out["flow_encoder_us_per_call"] = {"reference_sequence": fe["reference_sequence"] +
                                           f", {fe['launches']} launches",
                                           "exec_replay": round(fe["exec_replay_us_per_call"], 2)}
    if "hift_decode" in details:
        hd = details["hift_decode"]
        out["hift_decode_us_per_call"] = {"reference_sequence": hd["reference_sequence"] +
                                          f", {hd['launches']} launches",
                                          "exec_replay": round(hd["exec_replay_us_per_decode"], 2),
                                          "conv_TFLOPs": round(hd["conv_TFLOPs"], 1)}
    out["details"] = details
    if not a.no_cpu:
        out["cpu_baseline"] = cpu_baseline(W, a.cpu_seconds)
    else:
        out["cpu_baseline"] = None
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
