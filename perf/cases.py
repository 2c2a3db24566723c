"""The work this framework is timed on: LLaMA-2 token steps and operator blocks, through the public C API.

Sizes are those of the repository's own workloads (bench.py): the tiny decoder (dim 288, 6 layers), and slices of a few
layers at the 7B (dim 4096, 32 heads of 128, FFN 11008) and 13B (dim 5120, 40 heads, FFN 13824) widths. Five kinds:

  decode     greedy single-token steps through vkllm_hip_token_loop from a filled KV cache
  prompt     one prompt step (tensor_new -> build_graph -> graph_init -> upload -> graph_run -> read the ids)
  attention  a graph of VKLLM_OP_* nodes over projected Q, K, V: RoPE, cache rows, scores, masked softmax, P.V, heads
             concatenated (the nodes vkllm_llama2_build_self_attn_layer makes)
  mlp        a graph of RMSNORM, FFN_UP_AND_GATE, MATMUL and the residual BIN
  head       a graph of RMSNORM, the vocabulary MATMUL and ARG_MAX

Weights are N(0, 0.02) in fp16 and norm weights near 1. The output matrix holds the embedding rows in another order, so
that the next token is decided by a margin, as a trained model's is, and not by the rounding of near ties.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vkllm.c_amd"))
import pyvkllm as V  # noqa: E402

EPS, THETA, STD = 1e-5, 10000.0, 0.02
SHAPES = {
    "tiny": dict(dim=288, heads=6, ffn=768, layers=6, ctx=256),
    "7b": dict(dim=4096, heads=32, ffn=11008, layers=4, ctx=4096),
    "13b": dict(dim=5120, heads=40, ffn=13824, layers=2, ctx=4096),
}
VOCAB = 32000
SLICE_VOCAB = 1000  # of the prompt steps: their layers are what is measured, the vocabulary product is a case of its own


def listed():
    return [
        # generating with the smallest model: 32 launches of a few microseconds a token
        {"name": "tiny_decode", "kind": "decode", "shape": "tiny", "pos": 16, "steps": 16},
        # its prompt: the smallest call
        {"name": "tiny_prompt", "kind": "prompt", "shape": "tiny", "tokens": 16, "offset": 0},
        # generating right after a 128-token prompt: bound by reading the weights
        {"name": "decode_7b", "kind": "decode", "shape": "7b", "pos": 128, "steps": 16},
        # generating deep into a conversation: the cache reads count
        {"name": "decode_7b_far", "kind": "decode", "shape": "7b", "pos": 3583, "steps": 8},
        # a short question of odd length
        {"name": "prompt_7b_37", "kind": "prompt", "shape": "7b", "tokens": 37, "offset": 0},
        # the headline workload's prompt
        {"name": "prompt_7b_128", "kind": "prompt", "shape": "7b", "tokens": 128, "offset": 0},
        # the next message of a conversation: a ragged chunk behind 700 cached positions
        {"name": "prompt_7b_chunk", "kind": "prompt", "shape": "7b", "tokens": 301, "offset": 700},
        # a long prompt
        {"name": "prompt_7b_1024", "kind": "prompt", "shape": "7b", "tokens": 1024, "offset": 0},
        # a long prompt of the largest model
        {"name": "prompt_13b_2048", "kind": "prompt", "shape": "13b", "tokens": 2048, "offset": 0},
        # a program's own graph of operators: the attention layer of a 512-token prompt
        {"name": "attention_512", "kind": "attention", "shape": "7b", "tokens": 512, "offset": 0},
        # and its feed-forward layer
        {"name": "mlp_512", "kind": "mlp", "shape": "7b", "tokens": 512},
        # the vocabulary head of one generated token
        {"name": "head_1", "kind": "head", "shape": "7b", "tokens": 1},
    ]


def log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "prompt", "prompt", "attention", "mlp", "head"])
    shape = rng.choice(["tiny", "7b", "7b", "13b"])
    if kind == "decode":
        steps = rng.randint(4, 16)
        return {"kind": kind, "shape": shape, "pos": log_int(rng, 2, (256 if shape == "tiny" else 4000) - 20),
                "steps": steps}
    if kind == "prompt":
        top = 200 if shape == "tiny" else 2048 if shape == "13b" else 1500
        tokens = log_int(rng, 2, top)
        room = SHAPES[shape]["ctx"] - tokens
        return {"kind": kind, "shape": shape, "tokens": tokens,
                "offset": rng.choice([0, log_int(rng, 1, min(room, 1000))])}
    if kind == "attention":
        tokens = log_int(rng, 2, 200 if shape == "tiny" else 640)
        return {"kind": kind, "shape": shape, "tokens": tokens,
                "offset": rng.choice([0, rng.randint(1, 40 if shape == "tiny" else 640 - tokens + 1)])}
    if kind == "mlp":
        return {"kind": kind, "shape": shape, "tokens": log_int(rng, 1, 200 if shape == "tiny" else 384)}
    return {"kind": kind, "shape": shape, "tokens": log_int(rng, 1, 64)}


# ---- inputs, made from the seed alone ------------------------------------------------------------------------------
class Inputs:
    """Tensors of one seed, in the order in which they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed) * 7919 + 17)

    def half(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32).mul_(std).half()

    def norm(self, n):
        return 1.0 + 0.1 * torch.randn(n, generator=self.g, device="cuda", dtype=torch.float32)

    def ids(self, n, vocab):
        return torch.randint(0, vocab, (n,), generator=self.g, device="cuda", dtype=torch.int64)


def model_inputs(case, seed):
    s, x = SHAPES[case["shape"]], Inputs(seed)
    D, F = s["dim"], s["ffn"]
    vocab = VOCAB if case["kind"] == "decode" else SLICE_VOCAB
    m = {"vocab": vocab, "embd": x.half(vocab, D), "out_norm": x.norm(D), "layers": []}
    m["out"] = (torch.roll(m["embd"], 1, 0).float() * STD).half()  # token t is followed by token t + 1
    for _ in range(s["layers"]):
        m["layers"].append({"an": x.norm(D), "q": x.half(D, D, std=STD), "k": x.half(D, D, std=STD),
                            "v": x.half(D, D, std=STD), "o": x.half(D, D, std=STD), "fn": x.norm(D),
                            "u": x.half(F, D, std=STD), "g": x.half(F, D, std=STD), "d": x.half(D, F, std=STD)})
    before = case["pos"] if case["kind"] == "decode" else case["offset"]
    m["before"] = x.ids(before, vocab)  # the tokens whose keys and values are cached
    m["toks"] = x.ids(1 if case["kind"] == "decode" else case["tokens"], vocab)
    return m


def block_inputs(case, seed):
    s, x, S = SHAPES[case["shape"]], Inputs(seed), case["tokens"]
    D, F, H = s["dim"], s["ffn"], s["heads"]
    hd = D // H
    if case["kind"] == "attention":
        o = case["offset"]
        return {"q": x.half(1, 1, S, D, std=1.3), "k": x.half(1, 1, S, D, std=1.3), "v": x.half(1, 1, S, D, std=1.3),
                "kc": x.half(1, H, o + S, hd, std=1.3), "vc": x.half(1, H, o + S, hd, std=1.3)}
    if case["kind"] == "mlp":
        return {"x": x.half(1, 1, S, D), "norm": x.norm(D), "u": x.half(1, 1, F, D, std=STD),
                "g": x.half(1, 1, F, D, std=STD), "d": x.half(1, 1, D, F, std=STD)}
    w = x.half(1, 1, VOCAB, D, std=STD)
    rows = (w[0, 0, x.ids(S, VOCAB)].float() / STD + x.half(S, D).float()).half()  # rows with a decided next token
    return {"x": rows.view(1, 1, S, D), "norm": x.norm(D), "w": w}


# ---- what a program has in hand ------------------------------------------------------------------------------------
class DeviceArray:
    """A device address for torch.as_tensor; the tensor made of it keeps its owner."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (ptr, False), "version": 2,
                                         "strides": None}


TYPESTR = {V.F32: "<f4", V.F16: "<f2", V.U32: "<i4"}


def on_device(t, owner):
    """The memory of a (contiguous) framework tensor of the program `owner` as a torch tensor."""
    c = t.contents
    return torch.as_tensor(DeviceArray(c.data.dev, tuple(c.shapes), TYPESTR[c.dtype], owner), device="cuda")


class KvCache(ctypes.Structure):  # include/vkllm/vkllm_kvcache.h, its first fields
    _fields_ = [("kcaches", ctypes.POINTER(V.ArrayTensor)), ("vcaches", ctypes.POINTER(V.ArrayTensor))]


class Program:
    """A context and what was made on it, released together."""

    def __init__(self):
        self.ctx, self.model, self.graph, self.tensors = V.Ctx(0), None, None, []

    def __del__(self):
        if self.ctx.p is None:
            return
        self.ctx.sync()
        if self.graph is not None:
            V.lib().vkllm_graph_free(self.ctx.vp, self.graph)
        for t in self.tensors:
            self.ctx.free(t)
        if self.model is not None:
            self.model.close()
        self.ctx.close()

    # a graph of operators
    def begin(self):
        self.graph = ctypes.POINTER(V.Graph)()
        V.check("vkllm_graph_new", V.lib().vkllm_graph_new(self.ctx.vp, ctypes.byref(self.graph)))

    def add(self, t):
        V.check("vkllm_graph_add_node", V.lib().vkllm_graph_add_node(self.ctx.vp, self.graph, t))
        return t

    def input(self, x, dtype=V.F16, op=V.OP_NONE, srcs=(), params=None):
        t = self.add(self.ctx.tensor(list(x.shape), dtype, op=op, srcs=srcs, params=params))
        on_device(t, self).copy_(x)
        return t

    def op(self, op, shape, srcs, params=None, dtype=V.F16):
        return self.add(self.ctx.tensor(list(shape), dtype, op=op, srcs=list(srcs), params=params))

    def view(self, t, reshape=None, permute=None):
        r = V.TensorP()
        V.check("vkllm_tensor_copy_ref", V.lib().vkllm_tensor_copy_ref(self.ctx.vp, t, ctypes.byref(r)))
        self.add(r)
        for name, arg in (("vkllm_tensor_reshape", reshape), ("vkllm_tensor_permute", permute)):
            if arg is not None:
                V.check(name, getattr(V.lib(), name)(self.ctx.vp, r, (ctypes.c_uint32 * 4)(*arg)))
        return r

    def finish(self, output):
        L = V.lib()
        V.check("vkllm_graph_set_output", L.vkllm_graph_set_output(self.ctx.vp, self.graph, output))
        V.check("vkllm_graph_init", L.vkllm_graph_init(self.ctx.vp, self.graph))

    def run_graph(self):
        L = V.lib()
        V.check("vkllm_graph_run", L.vkllm_graph_run(self.ctx.vp, self.graph))
        V.check("vkllm_graph_post_run", L.vkllm_graph_post_run(self.ctx.vp, self.graph))


def prepare_model(case, seed):
    s, m, p = SHAPES[case["shape"]], model_inputs(case, seed), Program()
    p.model = V.Model(p.ctx, config=V.llama_config(s["layers"], s["dim"], s["heads"], s["ffn"], vocab=m["vocab"],
                                                   ctx=s["ctx"], eps=EPS, theta=THETA, std=STD), seed=0)
    w = p.model.m.weights
    pairs = [(w.tok_embed_weights, m["embd"]), (w.output_norm_weight, m["out_norm"]), (w.output_weight, m["out"])]
    for i, a in enumerate(m["layers"]):
        b = w.blocks.contents.data[i].contents
        pairs += [(b.attn_norm_weight, a["an"]), (b.ffn_norm_weight, a["fn"]), (b.WQ, a["q"]), (b.WK, a["k"]),
                  (b.WV, a["v"]), (b.WO, a["o"]), (b.WU, a["u"]), (b.WG, a["g"]), (b.WD, a["d"])]
    for t, x in pairs:
        on_device(t, p).view(-1).copy_(x.reshape(-1))
    torch.cuda.synchronize()
    toks, before = m["toks"].cpu().numpy().astype(np.uint32), m["before"].cpu().numpy().astype(np.uint32)
    if before.size:
        p.model.step(before, 0)
    decode = case["kind"] == "decode"
    end = case["pos"] + case["steps"] if decode else case["offset"] + case["tokens"]
    kv = ctypes.cast(w.kvcache, ctypes.POINTER(KvCache)).contents
    caches = [[on_device(c.contents.data[i], p)[0, :, :end] for i in range(s["layers"])] for c in (kv.kcaches, kv.vcaches)]
    logits = torch.zeros(1 if decode else case["tokens"], m["vocab"], dtype=torch.float16, pin_memory=True)
    return {"case": case, "program": p, "toks": toks, "caches": caches, "logits": logits}


def run_model(state):
    case, p, logits = state["case"], state["program"], state["logits"]
    if case["kind"] == "decode":
        ids = p.model.loop(state["toks"], case["steps"], case["pos"])[0]
    else:
        ids = p.model.step(state["toks"], case["offset"])
    V.check("vkllm_hip_model_last_logits", V.lib().vkllm_hip_model_last_logits(
        p.ctx.vp, ctypes.byref(p.model.m), logits.data_ptr(), logits.shape[0]))
    return {"ids": ids, "logits": logits, "k": state["caches"][0], "v": state["caches"][1]}


def prepare_block(case, seed):
    s, x, p, S = SHAPES[case["shape"]], block_inputs(case, seed), Program(), case["tokens"]
    D, F, H = s["dim"], s["ffn"], s["heads"]
    hd = D // H
    p.begin()
    plain = V.MatmulParams(1.0, 0)
    if case["kind"] == "attention":
        o = case["offset"]
        rope = V.RopeParams(o, THETA, False)
        split, axis, kv = (1, S, H, hd), (0, 2, 1, 3), o + S
        q, k, v = (p.view(p.input(x[n]), reshape=split, permute=axis) for n in ("q", "k", "v"))
        rq, rk = (p.op(V.OP_ROPE, (1, H, S, hd), [t], rope) for t in (q, k))
        kc, vc = (p.input(x[n], op=V.OP_UPDATE_ROWS, srcs=[t], params=V.UpdateRowsParams(o))
                  for n, t in (("kc", rk), ("vc", v)))
        scores = p.op(V.OP_MATMUL, (1, H, S, kv), [rq, p.view(kc)], V.MatmulParams(1.0 / math.sqrt(hd), 0))
        prob = p.op(V.OP_SOFTMAX, (1, H, S, kv), [scores], V.SoftmaxParams(1, o))
        out = p.op(V.OP_MATMUL, (1, H, S, hd), [prob, p.view(vc)], plain)
        heads = p.op(V.OP_COPY, split, [p.view(out, permute=axis)])
        p.finish(heads)
        return {"program": p, "out": {"heads": heads, "prob": prob, "kc": kc, "vc": vc}}
    if case["kind"] == "mlp":
        inp, n = p.input(x["x"]), p.input(x["norm"].view(1, 1, 1, D), V.F32)
        wu, wg, wd = (p.input(x[name]) for name in ("u", "g", "d"))
        norm = p.op(V.OP_RMSNORM, (1, 1, S, D), [inp, n], V.RmsnormParams(2.0, EPS))
        act = p.op(V.OP_FFN_UP_AND_GATE, (1, 1, S, F), [norm, wu, wg])
        down = p.op(V.OP_MATMUL, (1, 1, S, D), [act, wd], plain)
        y = p.op(V.OP_BIN, (1, 1, S, D), [inp, down], ctypes.c_int32(0))
        p.finish(y)
        return {"program": p, "out": {"act": act, "y": y}}
    inp, n, w = p.input(x["x"]), p.input(x["norm"].view(1, 1, 1, D), V.F32), p.input(x["w"])
    norm = p.op(V.OP_RMSNORM, (1, 1, S, D), [inp, n], V.RmsnormParams(2.0, EPS))
    logits = p.op(V.OP_MATMUL, (1, 1, S, VOCAB), [norm, w], plain)
    ids = p.op(V.OP_ARG_MAX, (1, 1, S, 1), [logits], dtype=V.U32)
    p.finish(ids)
    return {"program": p, "out": {"logits": logits, "ids": ids}}


def prepare(case, seed):
    if case["kind"] in ("decode", "prompt"):
        return prepare_model(case, seed)
    state = prepare_block(case, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    if "caches" in state:
        return run_model(state)
    state["program"].run_graph()
    if "seen" not in state:  # the outputs' memory exists from the first pass on
        state["seen"] = {n: on_device(t, state["program"]) for n, t in state["out"].items()}
    return state["seen"]


# ---- what a pass cannot do without ---------------------------------------------------------------------------------
def work(case):
    s = SHAPES[case["shape"]]
    D, F, L, H = s["dim"], s["ffn"], s["layers"], s["heads"]
    layer = 4 * D * D + 3 * D * F
    if case["kind"] == "decode":
        total = {"bytes": 0, "flops": 0}
        for kv in range(case["pos"] + 1, case["pos"] + case["steps"] + 1):
            total["bytes"] += 2 * (L * layer + VOCAB * D) + 4 * L * D * kv + 4 * L * D + 4 * D * (2 * L + 1) + 2 * VOCAB
            total["flops"] += 2 * (L * layer + VOCAB * D) + 4 * L * D * kv
        return total
    S = case["tokens"]
    if case["kind"] == "prompt":
        o = case["offset"]
        pairs = S * o + S * (S + 1) // 2
        return {"bytes": 2 * (L * layer + SLICE_VOCAB * D) + 4 * L * D * (o + 2 * S) + 4 * D * (2 * L + 1)
                + 2 * S * (D + SLICE_VOCAB),
                "flops": 2 * S * (L * layer + SLICE_VOCAB * D) + 4 * L * D * pairs}
    if case["kind"] == "attention":
        kv = case["offset"] + S
        # each operator's operands and result once: RoPE and cache rows of K, scores, probabilities, heads
        return {"bytes": 2 * (S * D * 4 + S * D * 4 + S * D + kv * D * 2 + 4 * H * S * kv + S * D * 3),
                "flops": 4 * D * S * kv}
    if case["kind"] == "mlp":
        return {"bytes": 2 * (3 * D * F + S * (8 * D + 2 * F)) + 4 * D, "flops": 6 * S * D * F}
    return {"bytes": 2 * (VOCAB * D + S * (3 * D + 2 * VOCAB)) + 4 * D + 4 * S, "flops": 2 * S * VOCAB * D}


def tolerance(case):
    # fp16 results of fp32 sums: a sum in another order lands on a neighbouring fp16 value now and then, and in a model
    # those differences travel through the layers that follow
    if case["kind"] in ("decode", "prompt"):
        return {"rel": 5e-3, "max": 0.1, "differ": 0.01}
    # attention: a score's neighbouring fp16 value (2^-8 at scores of 4 to 8) moves its probability by as much
    return {"rel": 2e-3, "max": 0.05, "differ": 0.01}


# ---- the same in 64 bits -------------------------------------------------------------------------------------------
def rms(x, w):
    return x * w.double() * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def rotate(x, offset):
    """RoPE on adjacent pairs of the last axis of [H, S, hd], row i at position offset + i."""
    hd, S = x.shape[-1], x.shape[-2]
    freq = THETA ** (torch.arange(0, hd, 2, device="cuda", dtype=torch.float64) / hd)
    angle = torch.arange(offset, offset + S, device="cuda", dtype=torch.float64)[:, None] / freq
    c, n, a, b = angle.cos(), angle.sin(), x[..., 0::2], x[..., 1::2]
    return torch.stack((c * a - n * b, n * a + c * b), -1).flatten(-2)


def softmax_rows(scores, offset):
    S, kv = scores.shape[-2:]
    later = torch.arange(kv, device="cuda")[None, :] > torch.arange(S, device="cuda")[:, None] + offset
    return torch.softmax(scores.masked_fill(later, -math.inf), -1)


def weighted(prob, v):
    """P.V; with as many cached positions as head dims the API's shape rule reads V transposed."""
    return prob @ (v.transpose(-1, -2) if v.shape[-2] == v.shape[-1] else v)


def exact_step(m, s, toks, kc, vc):
    """One step in 64 bits behind the cached rows kc, vc (lists of [H, kv, hd]); returns the logits, grows the caches."""
    D, H, S = s["dim"], s["heads"], toks.numel()
    hd, o = D // H, kc[0].shape[1]
    h = m["embd"][toks].double()
    for i, a in enumerate(m["layers"]):
        n = rms(h, a["an"])
        q, k, v = ((n @ a[w].double().T).view(S, H, hd).transpose(0, 1) for w in ("q", "k", "v"))
        kc[i], vc[i] = torch.cat((kc[i], rotate(k, o)), 1), torch.cat((vc[i], v), 1)
        q, att = rotate(q, o), torch.empty(S, H, hd, device="cuda", dtype=torch.float64)
        for j in range(0, H, 8):  # a few heads at a time: the scores are large
            part = slice(j, min(j + 8, H))
            prob = softmax_rows(q[part] @ kc[i][part].transpose(1, 2) / math.sqrt(hd), o)
            att[:, part] = weighted(prob, vc[i][part]).transpose(0, 1)
        h = h + att.view(S, D) @ a["o"].double().T
        n = rms(h, a["fn"])
        gate = n @ a["g"].double().T
        h = h + ((n @ a["u"].double().T) * gate * torch.sigmoid(gate)) @ a["d"].double().T
    return rms(h, m["out_norm"]) @ m["out"].double().T


def exact(case, seed):
    s = SHAPES[case["shape"]]
    if case["kind"] in ("decode", "prompt"):
        m = model_inputs(case, seed)
        empty = torch.empty(s["heads"], 0, s["dim"] // s["heads"], device="cuda", dtype=torch.float64)
        kc, vc = [empty] * s["layers"], [empty] * s["layers"]
        if m["before"].numel():
            exact_step(m, s, m["before"], kc, vc)
        toks, ids = m["toks"], []
        for _ in range(case.get("steps", 1)):
            logits = exact_step(m, s, toks, kc, vc)
            toks = logits.argmax(-1)
            ids.append(toks)
        return {"ids": torch.cat(ids), "logits": logits, "k": kc, "v": vc}
    x, S = {k: t.double() for k, t in block_inputs(case, seed).items()}, case["tokens"]
    if case["kind"] == "attention":
        D, H, o = s["dim"], s["heads"], case["offset"]
        q, k, v = (x[n].view(S, H, D // H).transpose(0, 1) for n in ("q", "k", "v"))
        kc, vc = x["kc"][0].clone(), x["vc"][0].clone()
        kc[:, o:], vc[:, o:] = rotate(k, o), v
        prob = softmax_rows(rotate(q, o) @ kc.transpose(1, 2) / math.sqrt(D // H), o)
        return {"heads": weighted(prob, vc).transpose(0, 1)[None], "prob": prob[None], "kc": kc[None], "vc": vc[None]}
    n = rms(x["x"][0, 0], x["norm"])
    if case["kind"] == "mlp":
        gate = n @ x["g"][0, 0].T
        act = (n @ x["u"][0, 0].T) * gate * torch.sigmoid(gate)
        return {"act": act[None, None], "y": (x["x"][0, 0] + act @ x["d"][0, 0].T)[None, None]}
    logits = n @ x["w"][0, 0].T
    return {"logits": logits[None, None], "ids": None}
