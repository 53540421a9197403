"""The calls that the framework's speed is measured on.

A case is a dict of plain values; prepare() makes what a program holds before
the call (inputs, prepared weights, a captured node list), run() is one pass
through the public entry points of chatterbox_amdvulkan_amd.cbxops, exact()
the same outputs from plain torch in float64.

Whole calls are node lists captured once and replayed, as the synthesis loops
do (one replay per utterance, flow step or token); the others are single
layers and blocks, called eagerly, as an op batch, or as a short node list.
"""
from __future__ import annotations

import math

import torch

from chatterbox_amdvulkan_amd import cbxops as C
from chatterbox_amdvulkan_amd import workloads as W
from chatterbox_amdvulkan_amd.cfm_estimator import CFMEstimator
from chatterbox_amdvulkan_amd.flow_encoder import FlowEncoderCall
from chatterbox_amdvulkan_amd.ggml_nodes import NodeList
from chatterbox_amdvulkan_amd.hift_decode import HiFTDecode, src_down_shape
from chatterbox_amdvulkan_amd.t3_decode import T3DecodeStep

# HiFT upsamplers: C_in -> (C_out, stride, kernel)
UPS = {512: (256, 8, 16), 256: (128, 5, 11), 128: (64, 3, 7)}
EST_MID, EST_TR = 2, 2         # resnets and transformers of the estimator case (the reference repeats them 12 and 4 times)
ENC_BLOCKS, ENC_UP = 3, 3      # conformer blocks of the flow encoder case (the reference: 6 and 4)


def listed():
    return [
        # a vocoder decode of 10 s of speech: the whole graph between the two host transforms
        {"name": "hift_decode", "kind": "hift", "T_mel": 500},
        # one vocoder resblock (three Snake -> conv -> Snake -> conv layers) of that decode's middle stage, odd length
        {"name": "resblock", "kind": "resblock", "ch": 128, "K": 7, "T": 19999},
        # the last upsampler of the same decode, called by itself
        {"name": "upsample", "kind": "upsample", "c_in": 128, "T": 20000},
        # the flow decoder's U-Net at the reference's 500 frames with a padded tail, two mid blocks
        {"name": "cfm_estimator", "kind": "cfm", "T": 500, "tail": 40},
        # its causal block by itself: masked causal conv, LayerNorm, Mish, mask
        {"name": "causal_block", "kind": "causal", "c_in": 512, "T": 500, "tail": 23},
        # group norms and LayerNorm + RoPE of a flow step over two guidance items, one launch
        {"name": "cfm_norms", "kind": "cfm_norms", "T": 500},
        # causal attention probabilities of a 512-token T3 prompt
        {"name": "scores_prefill", "kind": "scores", "form": "causal", "heads": 16, "q": 512, "n_past": 0},
        # embedding + first LayerNorm and a feed-forward GELU of that prompt, F16 tables
        {"name": "prefill", "kind": "prefill", "n": 512, "table": "f16"},
        # a token of the T3 decode loop: the list re-pointed, the token written, the replay
        {"name": "t3_token", "kind": "t3", "n_past": 255},
        # a decode step of 64 streams in F16 with a Q8_0 table: the smallest call
        {"name": "streams", "kind": "streams", "n": 64},
        # the flow encoder on 5 s of speech tokens, three blocks a stack
        {"name": "flow_encoder", "kind": "flow", "T": 125},
        # Snake on a batch of last-stage activations
        {"name": "snake_batch", "kind": "snake", "B": 16, "ch": 64, "T": 120000},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    k = rng.choice(["hift", "resblock", "resblock", "upsample", "cfm", "causal", "cfm_norms", "scores", "scores",
                    "prefill", "t3", "streams", "flow", "snake"])
    if k == "hift":
        return {"kind": k, "T_mel": _log(rng, 25, 480)}
    if k == "resblock":
        ch, K = rng.choice([256, 128, 64]), rng.choice([3, 7, 11])
        return {"kind": k, "ch": ch, "K": K, "T": _log(rng, 200, {256: 4000, 128: 20000, 64: 60001}[ch])}
    if k == "upsample":
        c = rng.choice([512, 256, 128])
        return {"kind": k, "c_in": c, "T": _log(rng, 25, {512: 500, 256: 4000, 128: 20000}[c])}
    if k == "cfm":
        T = _log(rng, 60, 1000)
        return {"kind": k, "T": T, "tail": rng.choice([0, T // 9])}
    if k == "causal":
        T = _log(rng, 60, 2000)
        return {"kind": k, "c_in": rng.choice([256, 320, 512]), "T": T, "tail": rng.choice([0, T // 7])}
    if k == "cfm_norms":
        return {"kind": k, "T": 4 * rng.randint(63, 150)}       # the op batch takes whole float4s of a channel
    if k == "scores":
        form = rng.choice(["causal", "plain", "sum"])
        return {"kind": k, "form": form, "heads": 16 if form == "causal" else 8, "q": _log(rng, 60, 1000),
                "n_past": rng.choice([0, rng.randint(1, 300)]) if form == "causal" else 0}
    if k == "prefill":
        return {"kind": k, "n": _log(rng, 30, 2000), "table": rng.choice(["f32", "f16", "q8_0"])}
    if k == "t3":
        return {"kind": k, "n_past": rng.randint(0, W.T3_MAX_CTX - 1)}
    if k == "streams":
        return {"kind": k, "n": _log(rng, 1, 256)}
    if k == "flow":
        return {"kind": k, "T": _log(rng, 30, 250)}
    return {"kind": k, "B": rng.choice([1, 1, 2, 4]), "ch": rng.choice([256, 128, 64]), "T": _log(rng, 2000, 60001)}


# ---- inputs -------------------------------------------------------------------

class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, mean=0.0, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda") * std + mean

    def alpha(self, ch):
        a = torch.rand((ch,), generator=self.g, device="cuda") + 0.5
        return a, 1.0 / (a + 1e-9)

    def ints(self, n, hi):
        return torch.randint(0, hi, (n,), generator=self.g, device="cuda", dtype=torch.int32)


def _mask(T, tail):
    m = torch.ones((T, 1), device="cuda")
    if tail:
        m[T - tail:] = 0.0
    return m


def _inputs(case, seed):
    """The input tensors of the cases that are not built by a node list class."""
    k, r = case["kind"], _Rand(seed)
    if k == "resblock":
        ch, K = case["ch"], case["K"]
        layers = []
        for _ in range(3):
            p = {}
            for i in ("1", "2"):
                p["a" + i], p["ai" + i] = r.alpha(ch)
                p["w" + i] = r.normal(ch, ch, K, std=1.0 / math.sqrt(ch * K))
                p["b" + i] = r.normal(ch, std=0.1)
            layers.append(p)
        return {"x": r.normal(case["T"], ch), "layers": layers}
    if k == "upsample":
        ci, (co, s, K) = case["c_in"], UPS[case["c_in"]]
        return {"x": r.normal(case["T"], ci), "w": r.normal(ci, co, K, std=1.0 / math.sqrt(ci * K / s)),
                "b": r.normal(co, std=0.1)}
    if k == "causal":
        ci = case["c_in"]
        return {"x": r.normal(case["T"], ci), "m": _mask(case["T"], case["tail"]),
                "w": r.normal(256, ci, 3, std=1.0 / math.sqrt(ci * 3)), "b": r.normal(256, std=0.1),
                "lw": r.normal(256, mean=1.0, std=0.05), "lb": r.normal(256, std=0.05)}
    if k == "cfm_norms":
        T, H = case["T"], W.CFM_HEADS * W.HEAD_DIM
        return {"x256": r.normal(2, 256, 1, T), "w256": r.normal(1, 256, 1, 1, mean=1.0, std=0.02),
                "b256": r.normal(1, 256, 1, 1, std=0.02),
                "x512": r.normal(2, 512, 1, T), "w512": r.normal(1, 512, 1, 1, mean=1.0, std=0.02),
                "b512": r.normal(1, 512, 1, 1, std=0.02),
                "xa": r.normal(2, T, H), "wa": r.normal(H, mean=1.0, std=0.02), "ba": r.normal(H, std=0.02)}
    if k == "scores":
        shape = (case["heads"], case["q"], case["q"] + case["n_past"])
        return {"a": r.normal(*shape, std=8.0), "b": r.normal(*shape, std=8.0) if case["form"] == "sum" else None}
    if k == "prefill":
        D = W.D_MODEL
        return {"table": r.normal(W.VOCAB, D, std=0.02), "pos": r.normal(W.VOCAB, D, std=0.02),
                "ids": r.ints(case["n"], W.VOCAB), "pos_ids": torch.arange(case["n"], dtype=torch.int32, device="cuda"),
                "w": r.normal(D, mean=1.0, std=0.02), "b": r.normal(D, std=0.02), "ffn": r.normal(case["n"], W.D_FF)}
    if k == "t3":
        L, D, F, H = W.T3_LAYERS, W.D_MODEL, W.D_FF, W.T3_HEADS
        d = {"speech_emb": r.normal(W.T3_SPEECH_VOCAB, D, std=0.02).half(),
             "pos_embd": r.normal(W.T3_POS_ROWS, D, std=0.02).half()}
        for n, width, mean, std in (("ln1_w", D, 1, .02), ("ln1_b", D, 0, .02), ("qkv_b", 3 * D, 0, .02),
                                    ("out_b", D, 0, .02), ("ln2_w", D, 1, .02), ("ln2_b", D, 0, .02),
                                    ("fc_b", F, 0, .02), ("proj_b", D, 0, .02), ("qkv_mm", 3 * D, 0, 1),
                                    ("kq", H * W.T3_MAX_CTX, 0, 3), ("out_mm", D, 0, .5), ("fc_mm", F, 0, 1),
                                    ("proj_mm", D, 0, .5)):
            d[n] = r.normal(L, width, mean=mean, std=std)
        d["out_w"], d["out_b_final"] = r.normal(D, mean=1.0, std=0.02), r.normal(D, std=0.02)
        d["token"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        d["position"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        return d
    if k == "streams":
        n, D = case["n"], W.D_MODEL
        return {"table": r.normal(W.VOCAB, D, std=0.02), "ids": r.ints(n, W.VOCAB), "x": r.normal(n, D).half(),
                "g": r.normal(D, mean=1.0, std=0.02), "q": r.normal(n, W.N_HEAD, W.HEAD_DIM).half(),
                "k": r.normal(n, W.N_HEAD, W.HEAD_DIM).half(), "pos": r.ints(n, 2048),
                "gate": r.normal(n, W.D_FF).half(), "up": r.normal(n, W.D_FF).half()}
    assert k == "snake"
    a, ai = r.alpha(case["ch"])
    return {"x": r.normal(case["B"], case["T"], case["ch"]), "a": a, "ai": ai}


def _q8(x):
    """Q8_0 blocks of x's rows (per 32: the F16 scale, then 32 signed bytes)."""
    rows, n = x.shape
    b = x.view(rows, n // 32, 32)
    d = (b.abs().amax(2) / 127.0)
    q = torch.round(b / d.clamp_min(1e-30)[:, :, None]).clamp(-127, 127).to(torch.int8)
    out = torch.empty((rows, n // 32, 34), dtype=torch.uint8, device=x.device)
    out[:, :, :2] = d.half().view(torch.uint8).view(rows, n // 32, 2)
    out[:, :, 2:] = q.view(torch.uint8)
    return out.view(rows, n // 32 * 34)


def _unq8(t, n):
    b = t.view(t.shape[0], n // 32, 34)
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    return (d * b[:, :, 2:].contiguous().view(torch.int8).double()).view(t.shape[0], n)


def _nan(*shape, dtype=torch.float32):
    return torch.full(shape, float("nan"), dtype=dtype, device="cuda")


# ---- prepare and run ------------------------------------------------------------

class _ListState:
    """A node list captured into an exec, and the tensors a caller reads after a replay."""

    def __init__(self, nodes, keep, convs=()):
        self.nodes, self.keep, self.convs = nodes, list(keep), list(convs)
        self.exec = nodes.g.capture(self.keep)
        self.out = [nodes.at(i) for i in self.keep]

    def __del__(self):
        self.exec.close()
        for c in self.convs:
            c.close()


def prepare(case, seed):
    k = case["kind"]
    if k in ("hift", "cfm", "flow"):
        if k == "hift":
            e = HiFTDecode(case["T_mel"], seed=seed)
        elif k == "cfm":
            e = CFMEstimator(case["T"], seed=seed, n_mid=EST_MID, n_tr=EST_TR, mask_tail=case["tail"])
        else:
            e = FlowEncoderCall(case["T"], seed=seed, n_blocks=ENC_BLOCKS, n_up_blocks=ENC_UP)
        return _ListState(e.b, e.keep, getattr(e, "convs", ()))
    i = _inputs(case, seed)
    if k == "resblock":
        b = NodeList(lambda shape, dtype: torch.full(shape, float("nan"), dtype=dtype, device="cuda"))
        x, convs = b.t(i["x"]), []
        for p, dil in zip(i["layers"], (1, 3, 5)):
            cw1, cw2 = C.Conv1dWeights(p["w1"]), C.Conv1dWeights(p["w2"])
            convs += [cw1, cw2]
            x = b.sublayer(x, {n: b.t(t) for n, t in p.items()}, dil, cw1, cw2)
        return _ListState(b, [x], convs)
    if k == "t3":
        st = T3DecodeStep(i, case["n_past"])
        return {"step": st, "exec": st.graph.capture(st.keep), "n_past": case["n_past"],
                "token": (seed * 2654435761 + 17) % W.T3_SPEECH_VOCAB}
    if k == "upsample":
        return {"i": i, "w": C.Conv1dWeights(i["w"], transpose_stride=UPS[case["c_in"]][1]), "up": UPS[case["c_in"]]}
    if k == "causal":
        return {"i": i, "w": C.Conv1dWeights(i["w"])}
    if k == "cfm_norms":
        pos = torch.arange(case["T"], dtype=torch.int32, device="cuda")
        rope = C.RopeCache(W.HEAD_DIM, n_pos=2048)
        out = [_nan(*i[n].shape) for n in ("x256", "x512", "xa")]
        ops = [C.Op(C.OP_GROUP_NORM, (i["x256"], i["w256"], i["b256"]), (out[0],), act=C.MISH, eps=1e-5, iparam=W.CFM_GROUPS),
               C.Op(C.OP_GROUP_NORM, (i["x512"], i["w512"], i["b512"]), (out[1],), act=C.MISH, eps=1e-5, iparam=W.CFM_GROUPS),
               C.Op(C.OP_LAYER_NORM_ROPE, (i["xa"], i["wa"], i["ba"], pos), (out[2],), eps=1e-5, rope=rope,
                    iparam=W.HEAD_DIM)]
        return {"i": i, "batch": C.OpBatch(ops), "out": out, "rope": rope, "pos": pos}
    if k == "prefill":
        n, D, q8 = case["n"], W.D_MODEL, case["table"] == "q8_0"
        tab = _q8(i["table"]) if q8 else i["table"].half() if case["table"] == "f16" else i["table"]
        pos = i["pos"].half() if case["table"] != "f32" else i["pos"]
        out = [_nan(n, D), _nan(n, D), _nan(n, W.D_FF)]
        ops = [C.Op(C.OP_GET_ROWS_ADD_LAYER_NORM, (tab, i["ids"], pos, i["pos_ids"], i["w"], i["b"]), (out[0], out[1]),
                    eps=W.LN_EPS, q8=(0,) if q8 else ()),
               C.Op(C.OP_UNARY, (i["ffn"],), (out[2],), act=C.GELU)]
        return {"i": i, "tab": tab, "pos": pos, "batch": C.OpBatch(ops), "out": out}
    if k == "streams":
        n, D = case["n"], W.D_MODEL
        tab, rope = _q8(i["table"]), C.RopeCache(W.HEAD_DIM, n_pos=2048)
        h = torch.float16
        out = [_nan(n, D, dtype=h), _nan(n, W.N_HEAD, W.HEAD_DIM, dtype=h), _nan(n, W.N_HEAD, W.HEAD_DIM, dtype=h),
               _nan(n, W.D_FF, dtype=h), _nan(n, D)]
        ops = [C.Op(C.OP_RMS_NORM, (i["x"], i["g"]), (out[0],), eps=1e-5),
               C.Op(C.OP_ROPE, (i["q"], i["pos"]), (out[1],), rope=rope),
               C.Op(C.OP_ROPE, (i["k"], i["pos"]), (out[2],), rope=rope),
               C.Op(C.OP_SWIGLU, (i["gate"], i["up"]), (out[3],)),
               C.Op(C.OP_GET_ROWS, (tab, i["ids"]), (out[4],), q8=(0,))]
        return {"i": i, "tab": tab, "batch": C.OpBatch(ops), "out": out, "rope": rope}
    return {"i": i, "case": dict(case)}


def run(state):
    if isinstance(state, _ListState):
        state.exec.launch()
        return state.out
    if "step" in state:
        st = state["step"]
        st.retarget(state["n_past"])
        st.set_token(state["token"], state["n_past"])
        state["exec"].update(keep=st.keep)
        state["exec"].launch()
        n = W.T3_HEADS * (state["n_past"] + 1)
        return {k: v[:, :n] if k == "probs" else v for k, v in st.out.items()}
    if "batch" in state:
        state["batch"].launch()
        return state["out"]
    i = state["i"]
    if "up" in state:
        _, s, K = state["up"]
        return C.conv_transpose1d(i["x"], state["w"], (K - s) // 2, C.CONV_PRO_LEAKY_RELU, slope=0.1, bias=i["b"])
    if "w" in state:
        h = C.causal_conv1d(i["x"], state["w"], mask=i["m"], bias=i["b"])
        return C.layer_norm_mask(h, i["lw"], i["lb"], 1e-5, i["m"], act=C.MISH, out=h)
    case = state["case"]
    if case["kind"] == "scores":
        sc = 1.0 / math.sqrt(W.HEAD_DIM)
        if case["form"] == "sum":
            return C.add_scale_diag_mask_soft_max(i["a"], i["b"], sc)
        return C.scale_diag_mask_soft_max(i["a"], sc, case["n_past"] if case["form"] == "causal" else -1)
    return C.snake(i["x"], i["a"], i["ai"])


# ---- what a pass cannot do without ------------------------------------------------

def work(case):
    k = case["kind"]
    if k == "hift":
        T = case["T_mel"]
        fr = (8 * T, 40 * T, 120 * T + 1)
        F = fr[2]
        flops = 2 * 512 * T * 80 * 7 + 2 * 18 * F * 64 * 7
        nbytes = 4 * (80 * T + 18 * F) + 2 * (512 * 80 * 7 + 64 * 18 * 7)   # mel, source; F16 weights
        out = 512 * T + 18 * F
        for f, ci, s, ks, t_in in zip(fr, (512, 256, 128), (15, 3, 1), (7, 7, 11), (T, 8 * T, 40 * T)):
            ch, _, K = UPS[ci]
            ksd = src_down_shape(s)[0]
            flops += 2 * ci * ch * K * t_in + 2 * ch * f * 18 * ksd + 12 * ch * ch * f * (ks + 21)
            nbytes += 2 * (ci * ch * K + 18 * ch * ksd + 6 * ch * ch * (ks + 21))
            out += 4 * ch * f                                               # the stage outputs a caller keeps
        out += 64 * F
        return {"bytes": nbytes + 4 * out, "flops": flops}
    if k == "resblock":
        ch, K, T = case["ch"], case["K"], case["T"]
        return {"bytes": 8 * T * ch + 6 * (2 * ch * ch * K + 12 * ch), "flops": 12 * T * ch * ch * K}
    if k == "upsample":
        ci, (co, s, K), T = case["c_in"], UPS[case["c_in"]], case["T"]
        return {"bytes": 4 * T * (ci + co * s) + 2 * ci * co * K, "flops": 2 * T * ci * co * K}
    if k == "cfm":
        T, res = case["T"], EST_MID + 2
        tr, ch = res * EST_TR, 256
        # per transformer: to_out, ff.2 in, two norms out; ff.0 in and out; scores in and out
        per_tr = T * (4 * ch + 2 * 1024) + 2 * 8 * T * T
        # per resnet: time MLP and res_conv outputs in, the masked input out (320, 256 or 512 channels)
        per_res = T * ch + 2 * 256 + 1024
        masked = T * (320 + EST_MID * ch + 512)
        wt = 2 * 3 * ch * (320 + 512 + EST_MID * ch + res * ch + 3 * ch)
        io = T * (4 * 80 + 320 * 0 + ch + 80 * 2) + 8 * 1024
        flops = 2 * T * 3 * ch * (320 + 512 + EST_MID * ch + res * ch + 3 * ch)
        return {"bytes": 4 * (tr * per_tr + res * per_res + masked + io) + wt, "flops": flops}
    if k == "causal":
        ci, T = case["c_in"], case["T"]
        return {"bytes": 4 * T * (ci + 256 + 1) + 2 * 3 * ci * 256, "flops": 2 * T * 3 * ci * 256}
    if k == "cfm_norms":
        n = 2 * case["T"] * (256 + 512 + W.CFM_HEADS * W.HEAD_DIM)
        return {"bytes": 8 * n, "flops": 12 * n}
    if k == "scores":
        n = case["heads"] * case["q"] * (case["q"] + case["n_past"])
        return {"bytes": 4 * n * (3 if case["form"] == "sum" else 2), "flops": 6 * n}
    if k == "prefill":
        n, D = case["n"], W.D_MODEL
        row = {"f32": 8 * D, "f16": 4 * D, "q8_0": D // 32 * 34 + 2 * D}[case["table"]]
        return {"bytes": n * (row + 8 + 8 * D + 8 * W.D_FF) + 8 * D, "flops": n * (10 * D + 20 * W.D_FF)}
    if k == "t3":
        b = W.t3_token_bytes(W.T3_LAYERS, case["n_past"])
        return {"bytes": b, "flops": 3 * b}
    if k == "streams":
        n, D = case["n"], W.D_MODEL
        return {"bytes": n * (4 * D + 8 * D + 6 * W.D_FF + D // 32 * 34 + 4 * D + 8) + 4 * D,
                "flops": n * (4 * D + 12 * D + 8 * W.D_FF + D)}
    if k == "flow":
        T, D, F, H = case["T"], 512, 2048, 8
        tot = 2 * T * D + 6 * T * D            # gather; embed linears (T and 2T): in, out
        tot += 2 * 2 * T * D + 4 * T * D + 2 * T * D + T * D   # conv biases in and out, layout copies in, the stack's output
        for n, t in ((ENC_BLOCKS, T), (ENC_UP, 2 * T)):
            tot += n * (t * D * 10 + 2 * t * F + 3 * H * t * t)  # v, k, q, out, w2 in; v, k, two q's, two norms out
        tot += 2 * T * D + 2 * 2 * T * 80
        return {"bytes": 4 * tot, "flops": 6 * tot}
    n = case["B"] * case["ch"] * case["T"]
    return {"bytes": 8 * n, "flops": 20 * n}


def tolerance(case):
    k = case["kind"]
    if k == "hift":
        return {"rel": 1e-2}       # F16 conv operands rounded anew in each of 60 convs in a row: 5e-3 from exact()
    if k == "resblock":
        return {"rel": 2e-3}       # six such convs: 7e-4 from exact()
    if k == "upsample":
        return {"rel": 5e-6}       # one conv: F32 sums of the same F16 products in another order
    if k == "cfm":
        return {"rel": 1e-3}       # one conv after another, their operands rounded to F16: 3e-4 from exact()
    if k == "causal":
        return {"rel": 1e-5}       # one conv, then a LayerNorm and Mish
    if k == "streams":
        return {"rel": 1e-3}       # F16 outputs: 2e-4 from exact()
    if k == "cfm_norms":
        return {"rel": 1e-5}       # F32 rotation angles: 3e-6 from exact()
    return {"rel": 1e-6}           # F32 arithmetic, 1e-7 from exact() (the F16 GELU table: the same values)


# ---- the same from plain torch in float64 -----------------------------------------

def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(0.79788456080286535587989211986876 * x * (1 + 0.044715 * x * x)))


def _mish(x):
    return x * torch.tanh(torch.nn.functional.softplus(x, threshold=40.0))


def _ln(x, eps):
    m = x.mean(-1, keepdim=True)
    d = x - m
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps)


def _conv(x, w, pad, dil, T_out, stride=1):
    """(T, C_in) with w (C_out, C_in, K), zero padding `pad` on the left."""
    co, ci, K = w.shape
    need = (T_out - 1) * stride + (K - 1) * dil + 1
    xp = torch.zeros((max(need, pad + x.shape[0]), ci), dtype=torch.float64, device=x.device)
    xp[pad:pad + x.shape[0]] = x
    y = torch.zeros((T_out, co), dtype=torch.float64, device=x.device)
    for j in range(K):
        y += xp[j * dil:j * dil + (T_out - 1) * stride + 1:stride] @ w[:, :, j].t().contiguous()
    return y


def _conv_t(x, w, stride):
    """The uncropped transposed conv: (T, C_in), w (C_in, C_out, K) -> ((T - 1) * stride + K, C_out)."""
    ci, co, K = w.shape
    T = x.shape[0]
    y = torch.zeros(((T - 1) * stride + K, co), dtype=torch.float64, device=x.device)
    for j in range(K):
        y[j:j + (T - 1) * stride + 1:stride] += x @ w[:, :, j].contiguous()
    return y


def _snake(x, a, ai):
    return x + torch.sin(x * a) ** 2 * ai


def _rope(x, pos):
    """NEOX rotation of x (..., n_tok, heads, 64) by the positions."""
    h = W.HEAD_DIM // 2
    th = pos.double()[:, None] * 10000.0 ** (-torch.arange(h, device=x.device, dtype=torch.float64) / h)
    c, s = torch.cos(th)[:, None], torch.sin(th)[:, None]
    a, b = x[..., :h], x[..., h:]
    return torch.cat((a * c - b * s, a * s + b * c), -1)


class _Shadow:
    """A node list evaluated in float64: every storage has a float64 copy, read
    and written through the tensors' shapes, strides and offsets."""

    def __init__(self, nodes):
        self.nodes, self.store = nodes, {}

    def view(self, i):
        t = self.nodes.at(i)
        key = t.untyped_storage().data_ptr()
        if key not in self.store:
            n = t.untyped_storage().nbytes() // t.element_size()
            flat = torch.as_strided(t, (n,), (1,), 0)
            self.store[key] = flat.double() if t.is_floating_point() else flat
        return torch.as_strided(self.store[key], t.shape, t.stride(), t.storage_offset())

    def run(self):
        for n in self.nodes.g.nodes:
            if n.op == C.GOP_VIEW:
                continue
            a = self.view(n.src[0])
            b = self.view(n.src[1]) if n.src[1] >= 0 else None
            d = self.view(n.dst)
            d.copy_(self.value(n, a, b).reshape(d.shape))

    def value(self, n, a, b):
        op = n.op
        if op == C.GOP_GET_ROWS:
            return a[b.long()]
        if op in (C.GOP_ADD, C.GOP_MUL):
            return a + b if op == C.GOP_ADD else a * b
        if op == C.GOP_SCALE:
            return a * n.fparam
        if op == C.GOP_NORM:
            return _ln(a, n.fparam)
        if op == C.GOP_SOFT_MAX:
            return torch.softmax(a * n.fparam, -1)
        if op == C.GOP_DIAG_MASK_INF:
            q, kv = a.shape[-2:]
            keep = torch.arange(kv, device=a.device)[None] <= n.iparam + torch.arange(q, device=a.device)[:, None]
            return torch.where(keep, a, float("-inf"))
        if op == C.GOP_UNARY:
            f = {C.GELU: _gelu, C.GELU_ERF: torch.nn.functional.gelu, C.SILU: torch.nn.functional.silu,
                 C.TANH: torch.tanh, C.SOFTPLUS: lambda x: torch.nn.functional.softplus(x, threshold=40.0),
                 C.SIN: torch.sin, C.SQR: torch.square}
            return f[n.iparam](a)
        if op == C.GOP_LEAKY_RELU:
            return torch.where(a > 0, a, a * n.fparam)
        if op == C.GOP_CPY:
            return a
        if op == C.GOP_CONCAT:
            return torch.cat((a, b), a.dim() - 1 - n.iparam)
        if op == C.GOP_IM2COL:
            stride, pad, dil = n.conv[0], n.conv[1], n.conv[2]
            K = a.shape[-1]
            x = torch.nn.functional.pad(b.reshape(b.shape[-2:]), (pad, pad))         # (C_in, T)
            T = self.nodes.at(n.dst).shape[-2]
            cols = [x[:, j * dil:j * dil + (T - 1) * stride + 1:stride] for j in range(K)]
            return torch.stack(cols, 1).permute(2, 0, 1).contiguous()                # (T, C_in, K)
        if op == C.GOP_MUL_MAT:
            return b.contiguous() @ a.t().contiguous()
        assert op == C.GOP_CONV_TRANSPOSE_1D
        return _conv_t(b.reshape(b.shape[-2:]).t().contiguous(), a.contiguous(), n.conv[0]).t()


def exact(case, seed):
    k = case["kind"]
    if k in ("hift", "cfm", "flow"):
        st = prepare(case, seed)
        sh = _Shadow(st.nodes)
        sh.run()
        return [sh.view(i).clone() for i in st.keep]
    if k == "t3":
        st = prepare(case, seed)
        s = st["step"]
        s.set_token(st["token"], st["n_past"])

        class L:        # the list's tensors and nodes under the names _Shadow reads
            g = s.graph

            @staticmethod
            def at(i):
                if any(i in ids for ids in s._kq_ids):
                    return g_views[i]
                return s.graph._torch[i]
        g_views = {}
        for il, ids in enumerate(s._kq_ids):
            for i, t in zip(ids, (s.dev["kq"], s._mid["s"], s._mid["mk"], s.out["probs"])):
                g_views[i] = s._scores(t, il, st["n_past"] + 1)
        sh = _Shadow(L)
        sh.run()
        n = W.T3_HEADS * (st["n_past"] + 1)
        res = {}
        for name, t in s.out.items():
            v = sh.store[t.untyped_storage().data_ptr()].view(t.shape)
            res[name] = v[:, :n] if name == "probs" else v
        return res
    i = _inputs(case, seed)
    d = {n: t.double() if isinstance(t, torch.Tensor) and t.is_floating_point() else t for n, t in i.items()}
    if k == "resblock":
        x, K = d["x"], case["K"]
        for p, dil in zip(i["layers"], (1, 3, 5)):
            p = {n: t.double() for n, t in p.items()}
            h = _conv(_snake(x, p["a1"], p["ai1"]), p["w1"], (K - 1) // 2 * dil, dil, x.shape[0]) + p["b1"]
            h = _conv(_snake(h, p["a2"], p["ai2"]), p["w2"], (K - 1) // 2, 1, x.shape[0]) + p["b2"]
            x = x + h
        return [x]
    if k == "upsample":
        _, s, K = UPS[case["c_in"]]
        y = _conv_t(torch.where(d["x"] > 0, d["x"], d["x"] * 0.1), d["w"], s)
        p = (K - s) // 2
        return y[p:y.shape[0] - p] + d["b"]
    if k == "causal":
        y = _conv(d["x"] * d["m"], d["w"], 2, 1, case["T"]) + d["b"]
        return _mish(_ln(y, 1e-5) * d["lw"] + d["lb"]) * d["m"]
    if k == "cfm_norms":
        out = []
        for n in ("256", "512"):
            x = d["x" + n]
            g = _ln(x.view(2, W.CFM_GROUPS, -1), 1e-5).view(x.shape)
            out.append(_mish(g * d["w" + n] + d["b" + n]))
        T = case["T"]
        y = (_ln(d["xa"], 1e-5) * d["wa"] + d["ba"]).view(2, T, W.CFM_HEADS, W.HEAD_DIM)
        out.append(_rope(y, torch.arange(T, device="cuda")).view(2, T, -1))
        return out
    if k == "scores":
        x = (d["a"] + d["b"] if d["b"] is not None else d["a"]) / math.sqrt(W.HEAD_DIM)
        if case["form"] == "causal":
            q, kv = x.shape[-2:]
            keep = torch.arange(kv, device="cuda")[None] <= case["n_past"] + torch.arange(q, device="cuda")[:, None]
            x = torch.where(keep, x, float("-inf"))
        return torch.softmax(x, -1)
    if k == "prefill":
        t = case["table"]
        tab = _unq8(_q8(i["table"]), W.D_MODEL) if t == "q8_0" else i["table"].half().double() if t == "f16" else d["table"]
        pos = i["pos"].half().double() if t != "f32" else d["pos"]
        h = tab[i["ids"].long()] + pos[i["pos_ids"].long()]
        return [h, _ln(h, W.LN_EPS) * d["w"] + d["b"], _gelu(d["ffn"])]
    if k == "streams":
        x = d["x"]
        rms = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * d["g"]
        return [rms, _rope(d["q"], i["pos"]), _rope(d["k"], i["pos"]), torch.nn.functional.silu(d["gate"]) * d["up"],
                _unq8(_q8(i["table"]), W.D_MODEL)[i["ids"].long()]]
    return _snake(d["x"], d["a"], d["ai"])
