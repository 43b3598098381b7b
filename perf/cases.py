"""The work that the framework's speed is measured on: a list of cases over
the entry points of the decode and prefill paths, and a generator of more of
the same ranges.

  listed()              the cases
  draw(rng)             one more case of the same ranges
  prepare(case, seed)   inputs, uploaded weights and captured graphs
  run(state)            one pass through the public entry points
  work(case)            bytes and operations a pass cannot do without
  tolerance(case)       what another correct implementation may differ by
  exact(case, seed)     the same outputs in 64 bits, in plain torch

Weights are GGUF block bytes made on the device from the seed, centred around
zero as trained weights are; activations are normal with a few channels ten
times larger, as after a norm in a trained model.  A decode pass goes through
several layers with inputs of their own, as a token does, so that the weights
come from memory and not from a cache; the layers are copies of one upload,
which keeps prepare() short.  Decode passes are captured into a HIP graph once
and replayed, which is how a decode loop runs, unless a case says otherwise.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llmtoy-zig_amd"))

import llmtoy_amd as lt  # noqa: E402
from llmtoy_amd import hip  # noqa: E402
from llmtoy_amd import lib as ltlib  # noqa: E402

TYPES = {"f32": 0, "q8_0": 8, "q4_k": 12, "q6_k": 14, "q5_0": 6, "q5_1": 7, "q3_k": 11, "iq4_nl": 20}
ELEMS = {"f32": 1, "q8_0": 32, "q4_k": 256, "q6_k": 256, "q5_0": 32, "q5_1": 32, "q3_k": 256, "iq4_nl": 32}
BYTES = {"f32": 4, "q8_0": 34, "q4_k": 144, "q6_k": 210, "q5_0": 22, "q5_1": 24, "q3_k": 110, "iq4_nl": 18}
IQ4_NL = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]


# ------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: the norm of one token's residual, called eagerly
        {"name": "norm_one_row", "op": "norm", "rows": 1, "n": 2048, "add": False},
        # an attention or FFN projection of a decode step, 16 layers of it
        {"name": "matvec_q4k_square", "op": "matvec", "type": "q4_k", "rows": 4096, "cols": 4096, "layers": 16},
        # a Q8_0 projection whose sizes are no powers of two (d_model 2816)
        {"name": "matvec_q8_ragged", "op": "matvec", "type": "q8_0", "rows": 7001, "cols": 2816, "layers": 8},
        # the output head of a 262,144-word vocabulary, once a token
        {"name": "matvec_q6k_head", "op": "matvec", "type": "q6_k", "rows": 262144, "cols": 2816, "layers": 1},
        # the dense FFN of a small model (896 -> 4864 -> 896), 12 layers
        {"name": "ffn_q8", "op": "ffn", "gate": "q8_0", "down": "q8_0", "d_model": 896, "d_ffn": 4864, "act": "silu",
         "layers": 12},
        # decode of the 128-expert, top-8 layer: F32 router, Q4_K experts
        {"name": "moe_decode", "op": "moe", "experts": 128, "d_model": 2048, "d_expert": 768, "k": 8, "router": "f32",
         "gate": "q4_k", "down": "q4_k", "act": "silu", "norm_topk": True, "shared": 0, "layers": 8},
        # the Gemma4 block of a decode step with the APEX expert formats
        {"name": "gemma4_apex", "op": "gemma4", "experts": 128, "d_model": 2816, "d_expert": 704, "k": 8,
         "router": "q8_0", "gate": "q3_k", "down": "iq4_nl", "act": "gelu", "layers": 8},
        # the same kind of layer from its three parts, for a caller that does
        # its own work between routing and experts
        {"name": "moe_by_ids", "op": "moe_ops", "experts": 128, "d_model": 2048, "d_expert": 768, "k": 8,
         "router": "f32", "gate": "q4_k", "down": "q4_k", "act": "silu", "norm_topk": True, "layers": 8},
        # decode from host buffers: an engine that keeps its activations on
        # the host and sends only this layer to the GPU
        {"name": "moe_host", "op": "moe_host", "experts": 128, "d_model": 2048, "d_expert": 768, "k": 8,
         "router": "f32", "gate": "q4_k", "down": "q4_k", "act": "silu", "norm_topk": True, "shared": 0, "layers": 8},
        # a short prompt of an odd length
        {"name": "prefill_short", "op": "prefill", "tokens": 37, "experts": 128, "d_model": 2048, "d_expert": 768,
         "k": 8, "router": "f32", "act": "silu", "norm_topk": True, "zipf": True},
        # an ordinary prompt, experts in unequal demand
        {"name": "prefill_512", "op": "prefill", "tokens": 512, "experts": 128, "d_model": 2048, "d_expert": 768,
         "k": 8, "router": "f32", "act": "silu", "norm_topk": True, "zipf": True},
        # a batch of a long prompt, or several prompts' tokens together
        {"name": "prefill_1024", "op": "prefill", "tokens": 1024, "experts": 128, "d_model": 2048, "d_expert": 768,
         "k": 8, "router": "f32", "act": "silu", "norm_topk": True, "zipf": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _times(rng, step, lo, hi):
    """A multiple of step from lo to hi, over its logarithm."""
    return min(hi, max(lo, step * int(round(_log(rng, lo, hi) / step))))


def draw(rng):
    op = rng.choice(["norm", "matvec", "matvec", "matvec", "ffn", "moe", "moe", "gemma4", "moe_ops", "moe_host",
                     "prefill", "prefill", "prefill"])
    act = rng.choice(["silu", "gelu"])
    if op == "norm":
        n = _log(rng, 256, 8192)
        return {"op": op, "rows": _log(rng, 1, 1024), "n": n, "add": rng.random() < 0.5}
    if op == "matvec":
        kind = rng.choice([t for t in TYPES if t != "f32"])
        cols = _times(rng, max(ELEMS[kind], 64), 512, 4864 if ELEMS[kind] == 32 else 5120)
        row = cols // ELEMS[kind] * BYTES[kind]
        rows = min(_log(rng, 500, 160000), 400_000_000 // row)
        return {"op": op, "type": kind, "rows": rows, "cols": cols, "layers": max(1, min(16, 200_000_000 // (row * rows)))}
    if op == "ffn":
        gate, down = rng.choice([("q8_0", "q8_0"), ("q8_0", "q8_0"), ("q4_k", "q4_k"), ("q4_k", "q6_k")])
        step = 32 if gate == "q8_0" else 256
        d, f = _times(rng, step, 512, 4096), _times(rng, step, 1024, 8192)
        size = 2 * f * (d // ELEMS[gate] * BYTES[gate]) + d * (f // ELEMS[down] * BYTES[down])
        return {"op": op, "gate": gate, "down": down, "d_model": d, "d_ffn": f, "act": act,
                "layers": max(1, min(12, 200_000_000 // size))}
    if op == "prefill":
        return {"op": op, "tokens": _log(rng, 3, 1024), "experts": rng.choice([32, 64, 100, 128]),
                "d_model": 256 * rng.randint(4, 8), "d_expert": 64 * rng.randint(6, 12), "k": rng.choice([2, 4, 6, 8]),
                "router": rng.choice(["f32", "f32", "q8_0"]), "act": act, "norm_topk": rng.random() < 0.7,
                "zipf": rng.random() < 0.6}
    d, f = 256 * rng.randint(4, 11), 32 * rng.randint(16, 32)
    case = {"op": op, "experts": rng.choice([32, 60, 64, 128, 160]), "d_model": d, "d_expert": f,
            "k": rng.choice([2, 4, 6, 8]), "router": rng.choice(["f32", "q8_0"]), "act": act}
    case["gate"], case["down"] = rng.choice([("q4_k", "q4_k"), ("q4_k", "q4_k"), ("q3_k", "iq4_nl"), ("q3_k", "q5_1"),
                                             ("q4_k", "q5_0")])
    if op == "gemma4":
        case["router"] = "q8_0"
    else:
        case["norm_topk"] = rng.random() < 0.7
        if op != "moe_ops":
            case["shared"] = 32 * rng.randint(16, 80) if rng.random() < 0.3 else 0
    case["layers"] = rng.randint(3, 8)
    return case


# ------------------------------------------------------------------- the inputs
def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1_000_003 + what) & 0x7FFFFFFF)
    return g


def _normal(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * scale


def _activations(g, rows, n):
    x = _normal(g, rows, n)
    big = torch.rand(n, generator=g, device="cuda") < 0.004
    return torch.where(big, x * 10.0, x).contiguous()


def _f16(v):
    return v.to(torch.float16).view(torch.uint8)


def _blocks(g, kind, rows, cols, valid=None):
    """uint8 [rows, row bytes] of random GGUF blocks of weights of about 0.03;
    the columns from `valid` on are zero."""
    if kind == "f32":
        return _normal(g, rows, cols, scale=0.02).view(torch.uint8)
    nb, bb = cols // ELEMS[kind], BYTES[kind]
    b = torch.randint(0, 256, (rows, nb, bb), generator=g, device="cuda", dtype=torch.uint8)
    s = (_normal(g, rows, nb, 1) * 0.3).exp()  # the spread of the blocks' scales

    def put(at, v):
        b[..., at:at + 2] = _f16(v)

    if kind == "q8_0":
        put(0, s * 4e-4)
    elif kind == "q4_k":
        put(0, s * 2e-4)
        put(2, s * 2e-4 * 7.5)
    elif kind == "q6_k":
        put(208, s * 4e-5)
    elif kind == "q5_0":
        put(0, s * 3e-3)
    elif kind == "q5_1":
        put(0, s * 3e-3)
        put(2, s * -16 * 3e-3)
    elif kind == "iq4_nl":
        put(0, s * 5e-4)
    elif kind == "q3_k":
        put(108, s * 7e-4)
    if valid is not None and valid < cols:
        if kind == "q4_k":  # by sub-blocks of 32: scale and minimum zero
            for j in range(valid // 32, cols // 32):
                sc = b[:, j // 8, 4:16]
                j %= 8
                if j < 4:
                    sc[:, j] &= 0xC0
                    sc[:, j + 4] &= 0xC0
                else:
                    sc[:, j + 4] = 0
                    sc[:, j - 4] &= 0x3F
                    sc[:, j] &= 0x3F
        else:
            b[:, valid // ELEMS[kind]:] = 0
    return b.view(rows, nb * bb)


def _down_cols(case):
    step = ELEMS[case.get("down", "q4_k")]
    return -(-case["d_expert"] // step) * step


def _inputs(case, seed):
    """Everything a pass of the case is made of, as device tensors."""
    op = case["op"]
    g, gx = _gen(seed, 1), _gen(seed, 2)
    if op == "norm":
        r, n = case["rows"], case["n"]
        return {"x": _activations(gx, r, n), "b": _normal(gx, r, n), "w": 1 + 0.2 * _normal(gx, n)}
    if op == "matvec":
        return {"w": _blocks(g, case["type"], case["rows"], case["cols"]),
                "x": _activations(gx, case["layers"], case["cols"])}
    if op == "ffn":
        d, f = case["d_model"], case["d_ffn"]
        return {"wg": _blocks(g, case["gate"], f, d), "wu": _blocks(g, case["gate"], f, d),
                "wd": _blocks(g, case["down"], d, f), "x": _activations(gx, case["layers"], d)}
    e, d, f = case["experts"], case["d_model"], case["d_expert"]
    kd = _down_cols(case)
    v = {"router": _blocks(g, case["router"], e, d), "gu": _blocks(g, case.get("gate", "q4_k"), e * 2 * f, d),
         "dn": _blocks(g, case.get("down", "q4_k"), e * d, kd, f)}
    if op == "prefill":
        v["x"] = _activations(gx, case["tokens"], d)
        if case["zipf"]:
            rank = torch.randperm(e, generator=gx, device="cuda") + 1
            v["bias"] = -1.1 * rank.float().log()
        return v
    v["x"] = _activations(gx, case["layers"], d)
    if case.get("shared"):
        s = case["shared"]
        v["sg"], v["su"], v["sd"] = _blocks(g, "q8_0", s, d), _blocks(g, "q8_0", s, d), _blocks(g, "q8_0", d, s)
    if op == "gemma4":
        v["dense"] = _normal(gx, case["layers"], d)
        for name, n in (("pre_ffw_norm_2", d), ("router_scale", d), ("down_exps_scale", e), ("post_ffw_norm_2", d),
                        ("post_ffw_norm", d)):
            v[name] = 1 + 0.2 * _normal(gx, n)
    return v


# ------------------------------------------------------------------- a pass
_context = []


def _ctx():
    if not _context:
        _context.append(lt.Context(0))
    return _context[0]


class State:
    """What a program has in hand before the call; gives its weights back."""

    def __init__(self, case):
        self.case, self.ctx, self.tensors, self.graph = case, _ctx(), [], None

    def upload(self, blocks, kind, rows, cols, n_experts=1):
        t = self.ctx.upload(blocks.cpu().numpy(), TYPES[kind], rows, cols, n_experts)
        self.tensors.append(t)
        return t

    def layers(self, *first):
        """One tuple of weights per layer: the uploads, then copies of them."""
        got = [first]
        for _ in range(self.case["layers"] - 1):
            got.append(tuple(t.clone() if t is not None else None for t in first))
            self.tensors += [t for t in got[-1] if t is not None]
        return got

    def capture(self):
        self.once()  # sizes the context's scratch
        self.ctx.sync()
        self.graph = hip.Graph(self.ctx.stream, self.once)

    def __del__(self):
        torch.cuda.synchronize()
        if self.graph is not None:
            self.graph.destroy()
        for t in self.tensors:
            t.free()


def _act(case):
    return ltlib.ACT_SILU if case["act"] == "silu" else ltlib.ACT_GELU_TANH


def prepare(case, seed):
    op, v, s = case["op"], _inputs(case, seed), State(case)
    ctx = s.ctx
    if op == "norm":
        x, b, w = v["x"], v["b"], v["w"]
        out = torch.zeros_like(x)
        s.once = (lambda: ltlib.add_rmsnorm(ctx, out, x, b, w)) if case["add"] else (lambda: ltlib.rmsnorm(ctx, out, x, w))
        s.out = out
        torch.cuda.synchronize()
        return s
    if op == "matvec":
        ws = s.layers(s.upload(v["w"], case["type"], case["rows"], case["cols"]))
        x = v["x"]
        s.out = torch.zeros(case["layers"], case["rows"], device="cuda")
        io = [(w[0], x[i], s.out[i]) for i, w in enumerate(ws)]

        def once():
            for w, xi, oi in io:
                ctx.quant_matvec(oi, w, xi)
    elif op == "ffn":
        d, f = case["d_model"], case["d_ffn"]
        ws = s.layers(s.upload(v["wg"], case["gate"], f, d), s.upload(v["wu"], case["gate"], f, d),
                      s.upload(v["wd"], case["down"], d, f))
        s.out = torch.zeros(case["layers"], d, device="cuda")
        io = [(w, v["x"][i], s.out[i]) for i, w in enumerate(ws)]
        act = _act(case)

        def once():
            for w, xi, oi in io:
                ctx.ffn_dense(oi, *w, xi, act=act)
    else:
        once = _prepare_moe(case, s, v)
    s.once = once
    torch.cuda.synchronize()
    if op == "prefill" or op == "moe_host" or case.get("layers") == 1:
        return s
    s.capture()
    return s


def _prepare_moe(case, s, v):
    op, ctx = case["op"], s.ctx
    e, d, f, k, kd = case["experts"], case["d_model"], case["d_expert"], case["k"], _down_cols(case)
    router = s.upload(v["router"], case["router"], e, d)
    gu = s.upload(v["gu"], case.get("gate", "q4_k"), 2 * f, d, e)
    dn = s.upload(v["dn"], case.get("down", "q4_k"), d, kd, e)
    act, norm = _act(case), bool(case.get("norm_topk"))
    if op == "prefill":
        x, bias = v["x"], v.get("bias")
        s.out = torch.zeros_like(x)
        return lambda: ctx.moe_prefill(s.out, x, router, gu, dn, k, f, act=act, norm_topk=norm, bias=bias)
    shared = [None] * 3
    if case.get("shared"):
        sh = case["shared"]
        shared = [s.upload(v["sg"], "q8_0", sh, d), s.upload(v["su"], "q8_0", sh, d), s.upload(v["sd"], "q8_0", d, sh)]
    ws, n = s.layers(router, gu, dn, *shared), case["layers"]
    if op == "moe_host":
        xs = v["x"].cpu().numpy()
        s.out = np.zeros((n, d), np.float32)
        outs = s.out
    else:
        xs = v["x"]
        s.out = outs = torch.zeros(n, d, device="cuda")
    if op == "gemma4":
        x0, x, dense = v["x"], s.out, v["dense"]
        norms = {q: v[q] for q in ("pre_ffw_norm_2", "router_scale", "down_exps_scale", "post_ffw_norm_2",
                                   "post_ffw_norm")}
        rows = [(x[i], dense[i], w) for i, w in enumerate(ws)]
        nbytes = x.numel() * 4

        def once():
            # the residual stream is updated in place: a fresh one for the pass
            hip.check(hip.hip().hipMemcpyAsync(x.data_ptr(), x0.data_ptr(), nbytes, hip.D2D, ctypes.c_void_p(ctx.stream)))
            for xi, di, w in rows:
                ltlib.gemma4_moe_block(ctx, xi, di, *w[:3], k, f, norms, layer_output_scale=0.75, act=act)
        return once
    if op == "moe_ops":
        ids = torch.zeros(n, k, dtype=torch.int32, device="cuda")
        p = torch.zeros(n, k, device="cuda")
        h = torch.zeros(n, k, kd, device="cuda")
        rows = [(xs[i], ids[i], p[i], h[i], outs[i], w) for i, w in enumerate(ws)]
        s.out = {"ids": ids, "weights": p, "h": h[..., :f], "out": outs}

        def once():
            for xi, ii, pi, hi, oi, w in rows:
                ctx.router_topk(w[0], xi, k, ii, pi, norm_topk=norm)
                ctx.expert_gate_up_id(w[1], xi, ii, k, f, kd, hi, act=act)
                ctx.expert_down_id(w[2], hi, ii, pi, k, oi)
        return once
    rows = [(xs[i], outs[i], w) for i, w in enumerate(ws)]

    def once():
        for xi, oi, w in rows:
            ctx.moe_forward(oi, xi, w[0], w[1], w[2], k, f, act=act, norm_topk=norm,
                            shared=w[3:] if w[3] is not None else None)
    return once


def run(state):
    if state.graph is not None:
        state.graph.launch()
    else:
        state.once()
    return state.out


# ------------------------------------------------------------------- what a pass needs
def _row_bytes(kind, cols):
    return cols // ELEMS[kind] * BYTES[kind]


def work(case):
    op = case["op"]
    if op == "norm":
        n = case["rows"] * case["n"]
        return {"bytes": 4 * (n * (3 if case["add"] else 2) + case["n"]), "flops": 4 * n}
    if op == "matvec":
        r, c = case["rows"], case["cols"]
        return {"bytes": case["layers"] * (r * _row_bytes(case["type"], c) + 4 * (r + c)),
                "flops": case["layers"] * 2 * r * c}
    d = case["d_model"]
    if op == "ffn":
        f = case["d_ffn"]
        return {"bytes": case["layers"] * (2 * f * _row_bytes(case["gate"], d) + d * _row_bytes(case["down"], f) + 8 * d),
                "flops": case["layers"] * 6 * d * f}
    e, f, k = case["experts"], case["d_expert"], case["k"]
    # the down rows' zero columns are no work a pass cannot do without
    kd = -(-f // ELEMS[case.get("down", "q4_k")]) * ELEMS[case.get("down", "q4_k")]
    expert = 2 * f * _row_bytes(case.get("gate", "q4_k"), d) + d * _row_bytes(case.get("down", "q4_k"), kd)
    route = e * _row_bytes(case["router"], d)
    if op == "prefill":
        t = case["tokens"]
        used = e * (1 - (1 - k / e) ** t)  # experts that equal demand would reach
        return {"bytes": used * expert + route + 8 * t * d, "flops": 6 * t * k * d * f + 2 * t * e * d}
    s = case.get("shared") or 0
    sh = 2 * s * _row_bytes("q8_0", d) + d * _row_bytes("q8_0", s)
    return {"bytes": case["layers"] * (k * expert + route + sh + 8 * d),
            "flops": case["layers"] * (6 * k * d * f + 2 * e * d + 6 * d * s)}


def tolerance(case):
    """About four times what two correct ways of computing differ by."""
    op = case["op"]
    if op == "norm":
        return {"rel": 1e-6, "max": 1e-5}
    if op == "prefill":  # f16 activations and weights in the experts' products: 8e-4 from 64 bits
        return {"rel": 3e-3, "max": 3e-2}
    if op == "matvec" and case["type"] == "q8_0" or op == "ffn" and case["gate"] == "q8_0":
        return {"rel": 1e-5, "max": 1e-4}  # 32-bit products and sums
    if op in ("matvec", "ffn"):  # activations in 16 bits of a group of 16's largest, or 32 bits: up to 5e-5
        return {"rel": 2e-4, "max": 2e-3}
    return {"rel": 4e-4, "max": 4e-3, "differ": 0.0}  # the same, through two products: up to 9e-5


# ------------------------------------------------------------------- the same in 64 bits
def _f64(b, at):
    return b[..., at:at + 2].contiguous().view(torch.float16).double()


def _decode(kind, blocks, cols):
    """float64 [rows, cols] of GGUF block bytes."""
    rows = blocks.shape[0]
    if kind == "f32":
        return blocks.contiguous().view(torch.float32).double().view(rows, cols)
    b = blocks.view(rows, cols // ELEMS[kind], BYTES[kind])
    if kind == "q8_0":
        v = _f64(b, 0) * b[..., 2:].contiguous().view(torch.int8).double()
    elif kind == "q4_k":
        s = b[..., 4:16].int()
        lo, hi, top = s[..., 0:4], s[..., 4:8], s[..., 8:12]
        sc = torch.cat([lo & 63, (top & 15) | (lo >> 6 << 4)], -1).double()
        mn = torch.cat([hi & 63, (top >> 4) | (hi >> 6 << 4)], -1).double()
        q = b[..., 16:].int().view(rows, -1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 3).view(rows, -1, 8, 32).double()
        v = (_f64(b, 0) * sc).unsqueeze(-1) * q - (_f64(b, 2) * mn).unsqueeze(-1)
    elif kind == "q6_k":
        ql, qh = b[..., 0:128].int().view(rows, -1, 2, 2, 32), b[..., 128:192].int().view(rows, -1, 2, 32)
        q = torch.stack([(ql[..., 0, :] & 15) | ((qh & 3) << 4), (ql[..., 1, :] & 15) | ((qh >> 2 & 3) << 4),
                         (ql[..., 0, :] >> 4) | ((qh >> 4 & 3) << 4), (ql[..., 1, :] >> 4) | (qh >> 6 << 4)], -2)
        sc = b[..., 192:208].contiguous().view(torch.int8).double().unsqueeze(-1)
        v = _f64(b, 208).unsqueeze(-1) * sc * (q.reshape(rows, -1, 16, 16).double() - 32)
    elif kind in ("q5_0", "q5_1"):
        at = 2 if kind == "q5_0" else 4
        h = b[..., at:at + 4].int()
        h = (h.unsqueeze(-1) >> torch.arange(8, device=b.device)) & 1
        h = h.reshape(rows, -1, 32)
        q = b[..., at + 4:].int()
        q = (torch.cat([q & 15, q >> 4], -1) | (h << 4)).double()
        v = _f64(b, 0) * (q - 16) if kind == "q5_0" else _f64(b, 0) * q + _f64(b, 2)
    elif kind == "iq4_nl":
        q = b[..., 2:].long()
        v = _f64(b, 0) * torch.tensor(IQ4_NL, device=b.device, dtype=torch.float64)[torch.cat([q & 15, q >> 4], -1)]
    else:  # q3_k
        hm, q, s = b[..., 0:32].int(), b[..., 32:96].int().view(rows, -1, 2, 1, 32), b[..., 96:108].int()
        sc = torch.cat([s[..., 0:4] & 15, s[..., 4:8] & 15, s[..., 0:4] >> 4, s[..., 4:8] >> 4], -1)
        top = torch.cat([s[..., 8:12] >> sh & 3 for sh in (0, 2, 4, 6)], -1)
        sc = (sc | (top << 4)).double() - 32
        two = (q >> torch.tensor([0, 2, 4, 6], device=b.device).view(4, 1)) & 3
        bit = (hm.unsqueeze(-2) >> torch.arange(8, device=b.device).view(8, 1)) & 1
        q = two.reshape(rows, -1, 8, 32) - 4 * (1 - bit)
        v = (_f64(b, 108) * sc).unsqueeze(-1) * q.reshape(rows, -1, 16, 16).double()
    return v.reshape(rows, cols)


def _activate(case, v):
    return torch.nn.functional.silu(v) if case["act"] == "silu" else torch.nn.functional.gelu(v, approximate="tanh")


def _routing(case, v, x):
    """(ids, weights) of the rows of x."""
    logits = x @ _decode(case["router"], v["router"], case["d_model"]).T
    if "bias" in v:
        logits = logits + v["bias"].double()
    p = logits.softmax(-1)
    ids = logits.topk(case["k"], -1).indices
    p = p.gather(-1, ids)
    return ids, p / p.sum(-1, keepdim=True) if case.get("norm_topk") else p


def _expert(case, v, e):
    """The expert's (gate, up, down) in 64 bits."""
    d, f, kd = case["d_model"], case["d_expert"], _down_cols(case)
    w = _decode(case.get("gate", "q4_k"), v["gu"][e * 2 * f:(e + 1) * 2 * f], d)
    return w[:f], w[f:], _decode(case.get("down", "q4_k"), v["dn"][e * d:(e + 1) * d], kd)[:, :f]


def _experts(case, v, x, ids, p, want_h=False):
    out = torch.zeros_like(x)
    h_all = torch.zeros(x.shape[0], case["k"], case["d_expert"], device=x.device, dtype=torch.float64)
    for e in ids.unique().tolist():
        t, s = (ids == e).nonzero(as_tuple=True)
        gate, up, down = _expert(case, v, e)
        h = _activate(case, x[t] @ gate.T) * (x[t] @ up.T)
        h_all[t, s] = h
        out.index_add_(0, t, p[t, s].unsqueeze(-1) * (h @ down.T))
    return (out, h_all) if want_h else out


def _rms(x, w, eps=1e-6):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w


def exact(case, seed):
    op, v = case["op"], _inputs(case, seed)
    x = v["x"].double()
    if op == "norm":
        return _rms(x + v["b"].double() if case["add"] else x, v["w"].double())
    if op == "matvec":
        part = max(1, 100_000_000 // case["cols"])
        rows = [x @ _decode(case["type"], w, case["cols"]).T for w in v["w"].split(part)]
        return torch.cat(rows, -1)
    d = case["d_model"]
    if op == "ffn":
        f = case["d_ffn"]
        h = _activate(case, x @ _decode(case["gate"], v["wg"], d).T) * (x @ _decode(case["gate"], v["wu"], d).T)
        return h @ _decode(case["down"], v["wd"], f).T
    if op == "gemma4":
        r_in = _rms(x, v["router_scale"].double()) / math.sqrt(d)
        ids, p = _routing(case, v, r_in)
        p = p * v["down_exps_scale"].double()[ids]
        moe = _experts(case, v, _rms(x, v["pre_ffw_norm_2"].double()), ids, p)
        c = v["dense"].double() + _rms(moe, v["post_ffw_norm_2"].double())
        return (x + _rms(c, v["post_ffw_norm"].double())) * 0.75
    ids, p = _routing(case, v, x)
    if op == "moe_ops":
        out, h = _experts(case, v, x, ids, p, True)
        return {"ids": None, "weights": p, "h": h, "out": out}
    out = _experts(case, v, x, ids, p)
    if case.get("shared"):
        s = case["shared"]
        h = _activate(case, x @ _decode("q8_0", v["sg"], d).T) * (x @ _decode("q8_0", v["su"], d).T)
        out = out + h @ _decode("q8_0", v["sd"], s).T
    return out
