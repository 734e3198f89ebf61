"""What a user of libkatali_hip has it do, as cases that can be timed.

Every case runs through the Python binding (katali-lab_amd/katali_hip.py): the
dense projections of a decode step, the MoE layer in its single-token, normed
and batched forms, the dense FFN, the LM head with greedy sampling, and one
whole decode token. A decode loop replays graphs, as INTEGRATION.md's engine
does per token; single calls run eagerly. Weights are Q4_K / Q6_K blocks of
uniform random quants whose super-block scales give a matrix of about
1/sqrt(cols) standard deviation, as trained weights have.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "katali-lab_amd"))
import katali_hip as K  # noqa: E402

Q4, Q6 = K.Q4_K, K.Q6_K
TYPES = {"q4": Q4, "q6": Q6}
DEV = "cuda"
EPS = 1e-6


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the steps before a MoE layer for an engine that needs the selection
        # itself (an expert tier): residual, norm and F32 router rows of a
        # 128-expert layer, then its top 8; two short launches
        {"name": "router_2048x128", "kind": "router", "hidden": 2048, "rows": 128, "sel": 8},
        # one Q4_K projection of a 2048-wide model against an activation
        # quantized once by its own call, as one that several share is
        {"name": "gemv_q4_6144x2048_q8", "kind": "gemv", "type": "q4", "rows": 6144, "cols": 2048, "act": "q8"},
        # q, k and v of a 4096-wide model in one call, the engine's default fp32 activation
        {"name": "qkv_4096_f32", "kind": "qkv", "cols": 4096, "q_rows": 4096, "kv_rows": 1024, "act": "f32"},
        # the down projection of a 5120-wide dense model, fp32 activation: long
        # rows of 54 super-blocks, no power of two
        {"name": "gemv_q6_5120x13824_f32", "kind": "gemv", "type": "q6", "rows": 5120, "cols": 13824, "act": "f32"},
        # one Q4_K projection of an odd number of rows, the activation quantized in the call
        {"name": "gemv_q4_9731x2560", "kind": "gemv", "type": "q4", "rows": 9731, "cols": 2560, "act": "dp4a"},
        # the LM head over a 151936-word vocabulary and the greedy token
        {"name": "head_151936x2048", "kind": "head", "rows": 151936, "cols": 2048, "act": "f32"},
        # 16 decode layers, top-8 of 128 experts routed on the device
        {"name": "moe_2048x768_8of128", "kind": "moe", "layers": 16, "hidden": 2048, "ffn": 768, "experts": 128,
         "sel": 8, "shared": False, "down": "q6", "route": "logits"},
        # 16 decode layers, top-8 of 256 small experts and a shared expert
        {"name": "moe_2048x512_8of256_sh", "kind": "moe", "layers": 16, "hidden": 2048, "ffn": 512, "experts": 256,
         "sel": 8, "shared": True, "down": "q6", "route": "logits"},
        # 2 decode layers of few wide experts, the selection given by the engine
        {"name": "moe_4096x14336_2of8", "kind": "moe", "layers": 2, "hidden": 4096, "ffn": 14336, "experts": 8,
         "sel": 2, "shared": False, "down": "q6", "route": "given"},
        # 4 dense decode layers (norms, q/k/v, o, SwiGLU FFN) of a 4096-wide model
        {"name": "dense_4096x12288", "kind": "dense", "layers": 4, "hidden": 4096, "q_rows": 4096, "kv_rows": 1024,
         "ffn": 12288, "act": "dp4a"},
        # a prompt chunk: 64 tokens routed and run through a top-8 of 128 layer
        {"name": "batch_64_8of128", "kind": "batch", "tokens": 64, "hidden": 2048, "ffn": 768, "experts": 128,
         "sel": 8, "shared": False, "down": "q6"},
        # one whole decode token, attention aside: 48 normed MoE layers, the
        # output norm, the LM head and the greedy token
        {"name": "token_48x2048", "kind": "token", "layers": 48, "hidden": 2048, "ffn": 768, "experts": 128,
         "sel": 8, "down": "q6", "rows": 151936},
    ]


def draw(rng):
    """One more case of the listed ones' ranges."""
    def logu(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def cols(lo, hi):
        return 256 * max(1, logu(lo, hi) // 256)

    kind = rng.choice(["router", "gemv", "gemv", "gemv", "qkv", "head", "moe", "moe", "moe", "dense", "batch",
                       "batch", "batch", "token"])
    act = rng.choice(["f32", "dp4a", "q8"])
    if kind == "router":
        rows = logu(8, 512)
        return {"kind": kind, "hidden": 4 * logu(64, 2048), "rows": rows, "sel": rng.randint(1, 8)}
    if kind == "gemv":
        c = cols(1024, 16384)
        return {"kind": kind, "type": rng.choice(["q4", "q6"]), "rows": logu(256, min(65536, 300000000 // c)), "cols": c,
                "act": act}
    if kind == "qkv":
        c = cols(1024, 8192)
        return {"kind": kind, "cols": c, "q_rows": 128 * logu(8, 64), "kv_rows": 128 * logu(1, 16),
                "act": rng.choice(["f32", "dp4a"])}
    if kind == "head":
        c = cols(1024, 5120)
        return {"kind": kind, "rows": logu(32000, 152000), "cols": c, "act": rng.choice(["f32", "dp4a"])}
    if kind == "dense":
        h = rng.choice([1024, 2048, 4096])
        return {"kind": kind, "layers": rng.randint(2, 4), "hidden": h, "q_rows": h,
                "kv_rows": 128 * rng.choice([2, 4, 8]), "ffn": cols(2 * h, 3.5 * h), "act": rng.choice(["f32", "dp4a"])}
    down = rng.choice(["q6", "q6", "q4"])
    if kind == "token":
        return {"kind": kind, "layers": rng.randint(4, 24), "hidden": rng.choice([1024, 2048]),
                "ffn": 256 * rng.randint(2, 4), "experts": rng.choice([32, 60, 64, 128]), "sel": rng.choice([4, 6, 8]),
                "down": down, "rows": logu(32000, 152000)}
    while True:
        hidden = rng.choice([1024, 2048, 2048, 4096])
        ffn = cols(256, 14336 if kind == "moe" else 4096)
        experts = rng.choice([8, 16, 32, 60, 64, 128, 160, 256])
        sel = rng.choice([1, 2, 4, 6, 8, 8, 8, 10])
        shared = rng.random() < 0.3
        slots = sel + shared
        if sel > experts or slots * ffn > 100000 or experts * hidden * ffn > 700e6:
            continue
        c = {"kind": kind, "hidden": hidden, "ffn": ffn, "experts": experts, "sel": sel, "shared": shared, "down": down}
        if kind == "moe":
            per = slots * hidden * ffn
            return dict(c, layers=max(1, min(16, int(160e6 / per), int(3.2e9 / (experts * hidden * ffn)))),
                        route=rng.choice(["logits", "logits", "given"]))
        return dict(c, tokens=logu(2, 64))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
_hip = None


def hip():
    global _hip
    if _hip is None:
        _hip = K.KataliHip()
        if not _hip.probe():
            raise RuntimeError(_hip.status())
    return _hip


class Buf:
    """A torch tensor on the GPU as the binding's buffers: it reads .ptr."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


class Inputs:
    """Random inputs, made in one order from the seed alone (prepare and exact
    draw the same ones)."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, device=DEV, generator=self.g) * std

    def weights(self, t, n, rows, cols):
        """n matrices of Q4_K or Q6_K blocks, [n][rows][cols / 256][block bytes]."""
        bb = K.BLOCK_BYTES[t]
        nblk = n * rows * (cols // 256)
        words = torch.empty((nblk * bb + 7) // 8, dtype=torch.int64, device=DEV)
        words.random_(-(2 ** 63), None, generator=self.g)
        b = words.view(torch.uint8)[:nblk * bb].view(nblk, bb)
        # the standard deviation of scale * quant is 322 d for Q4_K (6-bit
        # scales, 4-bit quants) and 1366 d for Q6_K (8-bit scales, 6-bit quants)
        sigma = 1.0 / ((322.0 if t == Q4 else 1366.0) * math.sqrt(cols))
        fields = (0, 2) if t == Q4 else (208,)
        for at in fields:
            d = (torch.randn(nblk, device=DEV, generator=self.g).abs_() * sigma).to(torch.float16)
            b[:, at:at + 2] = d.view(torch.uint8).view(nblk, 2)
        return b.view(n, rows, cols // 256, bb)


def experts(g, c, n):
    """gate, up [n][ffn][hidden], down [n][hidden][ffn]"""
    return (g.weights(Q4, n, c["ffn"], c["hidden"]), g.weights(Q4, n, c["ffn"], c["hidden"]),
            g.weights(TYPES[c["down"]], n, c["hidden"], c["ffn"]))


def logits(g, *shape):
    return g.normal(*shape)


def zipf_logits(g, tokens, n):
    """A prompt's router logits: an expert popularity common to its tokens
    (Zipf 1.1 over a random order) and a Gumbel draw per token."""
    order = torch.randperm(n, device=DEV, generator=g.g)
    pop = torch.empty(n, device=DEV)
    pop[order] = -1.1 * torch.log(torch.arange(1, n + 1, device=DEV, dtype=torch.float32))
    u = torch.rand(tokens, n, device=DEV, generator=g.g).clamp_(1e-7, 1 - 1e-7)
    return pop + -torch.log(-torch.log(u))


def inputs(c, seed):
    g, k = Inputs(seed), c["kind"]
    v = {}
    if k == "router":
        h = c["hidden"]
        v.update(x=g.normal(h), delta=g.normal(h), norm=1.0 + g.normal(h, std=0.1),
                 w=g.normal(c["rows"], h, std=1 / math.sqrt(h)))
    elif k in ("gemv", "head"):
        t = TYPES[c.get("type", "q6")]
        v.update(x=g.normal(c["cols"]), w=g.weights(t, 1, c["rows"], c["cols"])[0])
    elif k == "qkv":
        v.update(x=g.normal(c["cols"]), w=[g.weights(t, 1, r, c["cols"])[0] for t, r in qkv_mats(c)])
    elif k == "moe":
        v["layers"] = []
        for _ in range(c["layers"]):
            L = {"x": g.normal(c["hidden"]), "w": experts(g, c, c["experts"]), "logits": logits(g, c["experts"])}
            if c["shared"]:
                L["sh"] = experts(g, c, 1)
            v["layers"].append(L)
    elif k == "batch":
        v.update(x=g.normal(c["tokens"], c["hidden"]), w=experts(g, c, c["experts"]),
                 logits=zipf_logits(g, c["tokens"], c["experts"]))
        if c["shared"]:
            v["sh"] = experts(g, c, 1)
    elif k == "dense":
        h = c["hidden"]
        v["x"] = g.normal(h)
        v["layers"] = [{"n1": 1.0 + g.normal(h, std=0.1), "n2": 1.0 + g.normal(h, std=0.1),
                        "qkv": [g.weights(t, 1, r, h)[0] for t, r in qkv_mats(dict(c, cols=h))],
                        "o": g.weights(Q4, 1, h, c["q_rows"])[0], "ffn": experts(g, dict(c, down="q6"), 1)}
                       for _ in range(c["layers"])]
    else:
        h = c["hidden"]
        # a residual stream well above what one layer adds to it, as in
        # trained models
        v["x"] = g.normal(h, std=8.0)
        v["layers"] = [{"norm": 1.0 + g.normal(h, std=0.1), "router": g.normal(c["experts"], h, std=1 / math.sqrt(h)),
                        "w": experts(g, c, c["experts"])} for _ in range(c["layers"])]
        v.update(norm=1.0 + g.normal(h, std=0.1), head=g.weights(Q6, 1, c["rows"], h)[0])
    return v


def qkv_mats(c):
    return [(Q4, c["q_rows"]), (Q4, c["kv_rows"]), (Q6, c["kv_rows"])]


def given(lg, sel):
    """The selection an engine passes: top experts, largest first, and their
    softmax weights renormalised over the selection."""
    top, ids = torch.topk(lg.double(), sel, dim=-1)
    return ids.to(torch.int32), torch.softmax(top, dim=-1).float()


# ---------------------------------------------------------------------------
# the calls
# ---------------------------------------------------------------------------
class State:
    """What a program keeps between calls; a captured graph is given back with it."""

    def __init__(self, call, out, keep, graph=False):
        self.call, self.out, self.keep, self.graph = call, out, keep, None
        torch.cuda.synchronize()
        call()   # the library's scratch is allocated by the first call, outside any capture
        hip().sync()
        if graph:
            hip().graph_begin()
            call()
            self.graph = hip().graph_end()

    def __del__(self):
        if self.graph:
            hip().sync()
            hip().graph_destroy(self.graph)
            self.graph = None


def empty(*shape, dtype=torch.float32):
    return Buf(torch.zeros(*shape, device=DEV, dtype=dtype))


def matvec(t, w, rows, cols, x, y, act, xq):
    h = hip()
    if act == "f32":
        h.matvec(t, w, rows, cols, x, y)
    elif act == "dp4a":
        h.matvec_dp4a(t, w, rows, cols, x, y)
    else:
        h.quantize_q8_1(x, cols, xq)
        h.matvec_q8(t, w, rows, cols, xq, y)


def prepare(case, seed):
    c, h, k = case, hip(), case["kind"]
    v = inputs(c, seed)
    if k == "router":
        n, rows = c["hidden"], c["rows"]
        x, delta, norm, w = (Buf(v[i]) for i in ("x", "delta", "norm", "w"))
        xo, xn, y = empty(n), empty(n), empty(rows)
        ids, wts = empty(c["sel"], dtype=torch.int32), empty(c["sel"])

        def call():
            h.rmsnorm_matvec_f32(x, delta, 1.0, xo, norm, n, EPS, xn, w, rows, y)
            h.moe_route_batch(y, 1, rows, c["sel"], ids, wts)
        return State(call, [xo.t, xn.t, y.t, ids.t, wts.t], (x, delta, norm, w, xo, xn, y, ids, wts))
    if k in ("gemv", "head"):
        t, rows, cols = TYPES[c.get("type", "q6")], c["rows"], c["cols"]
        x, w, y = Buf(v["x"]), Buf(v["w"]), empty(rows)
        xq, tok = empty(cols // 32 * 36, dtype=torch.uint8), empty(1, dtype=torch.int32)

        def call():
            matvec(t, w, rows, cols, x, y, c["act"], xq)
            if k == "head":
                h.argmax(y, rows, tok)
        return State(call, [y.t, tok.t] if k == "head" else [y.t], (x, w, y, xq, tok))
    if k == "qkv":
        x, ws = Buf(v["x"]), [Buf(w) for w in v["w"]]
        types, rows = [m[0] for m in qkv_mats(c)], [m[1] for m in qkv_mats(c)]
        ys = [empty(r) for r in rows]

        def call():
            h.matvec_multi(types, ws, rows, c["cols"], x, ys, dp4a=c["act"] == "dp4a")
        return State(call, [y.t for y in ys], (x, ws, ys))
    if k == "moe":
        calls, out, keep = [], [], []
        for L in v["layers"]:
            w, x, y = [Buf(m) for m in L["w"]], Buf(L["x"]), empty(c["hidden"])
            sh = [Buf(m) for m in L["sh"]] if c["shared"] else None
            desc = h.moe_desc(c["hidden"], c["ffn"], c["experts"], *w, down_type=TYPES[c["down"]], shared=sh)
            if c["route"] == "logits":
                route = h.moe_route(c["sel"], logits=Buf(L["logits"]))
            else:
                ids, wts = given(L["logits"], c["sel"])
                route = h.moe_route(c["sel"], ids=Buf(ids), weights=Buf(wts))
            calls.append((desc, route, y, x))
            out.append(y.t)
            keep.append((w, sh, desc, route))

        def call():
            for desc, route, y, x in calls:
                h.moe_layer(desc, route, y, x=x)
        return State(call, out, keep, graph=True)
    if k == "batch":
        T, E, n = c["tokens"], c["experts"], c["sel"]
        w, x, lg, y = [Buf(m) for m in v["w"]], Buf(v["x"]), Buf(v["logits"]), empty(T, c["hidden"])
        sh = [Buf(m) for m in v["sh"]] if c["shared"] else None
        ids, wts = empty(T, n, dtype=torch.int32), empty(T, n)
        desc = h.moe_desc(c["hidden"], c["ffn"], E, *w, down_type=TYPES[c["down"]], shared=sh)

        def call():
            h.moe_route_batch(lg, T, E, n, ids, wts)
            h.moe_batch(desc, T, n, ids, wts, x, y)
        return State(call, [y.t], (w, x, lg, y, sh, ids, wts, desc))
    if k == "dense":
        n, qr, kr = c["hidden"], c["q_rows"], c["kv_rows"]
        types, rows = [Q4, Q4, Q6], [qr, kr, kr]
        x0, x, xn = Buf(v["x"]), empty(n), empty(n)
        route, layers, zero = h.moe_route(0), [], empty(n)
        for L in v["layers"]:
            ffn = [Buf(m) for m in L["ffn"]]
            layers.append({"n1": Buf(L["n1"]), "n2": Buf(L["n2"]), "qkv": [Buf(m) for m in L["qkv"]], "o": Buf(L["o"]),
                           "out": [empty(qr), empty(kr), empty(kr)], "y": empty(n), "att": empty(n),
                           "desc": h.moe_desc(n, c["ffn"], 0, None, None, None, shared=ffn), "ffn": ffn})

        def call():
            h.copy(x, x0, 4 * n)
            delta = zero
            for L in layers:
                h.add_rmsnorm(x, delta, 1.0, L["n1"], n, EPS, xn)
                h.matvec_multi(types, L["qkv"], rows, n, xn, L["out"], dp4a=c["act"] == "dp4a")
                matvec(Q4, L["o"], n, qr, L["out"][0], L["att"], c["act"], None)
                h.add_rmsnorm(x, L["att"], 1.0, L["n2"], n, EPS, xn)
                h.moe_layer(L["desc"], route, L["y"], x=xn)
                delta = L["y"]
        out = [t for L in layers for t in [o.t for o in L["out"]] + [L["att"].t, L["y"].t]]
        return State(call, out, (x0, x, xn, layers, route, zero), graph=True)
    # a whole token
    n, E, S = c["hidden"], c["experts"], c["sel"]
    x0, res = Buf(v["x"]), [empty(n), empty(n)]
    norm, head, xn, lg, tok = Buf(v["norm"]), Buf(v["head"]), empty(n), empty(c["rows"]), empty(1, dtype=torch.int32)
    layers = []
    for L in v["layers"]:
        w = [Buf(m) for m in L["w"]]
        layers.append((h.moe_desc(n, c["ffn"], E, *w, down_type=TYPES[c["down"]]), Buf(L["norm"]), Buf(L["router"]),
                       empty(n), w))

    def call():
        cur, delta = x0, None
        for i, (desc, nw, router, y, _) in enumerate(layers):
            h.moe_layer_normed(desc, S, cur, nw, router, y, delta=delta, x_out=res[i % 2], eps=EPS)
            if delta is not None:
                cur = res[i % 2]
            delta = y
        h.add_rmsnorm(cur, delta, 1.0, norm, n, EPS, xn)
        h.matvec_dp4a(Q6, head, c["rows"], n, xn, lg)
        h.argmax(lg, c["rows"], tok)
    return State(call, [layers[-1][3].t, lg.t, tok.t], (x0, res, norm, head, xn, lg, tok, layers), graph=True)


def run(state):
    if state.graph:
        hip().graph_launch(state.graph)
    else:
        state.call()
    return state.out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def wbytes(t, rows, cols):
    return rows * (cols // 256) * K.BLOCK_BYTES[t]


def expert_bytes(c):
    return 2 * wbytes(Q4, c["ffn"], c["hidden"]) + wbytes(TYPES[c.get("down", "q6")], c["hidden"], c["ffn"])


def distinct(c):
    """Distinct experts that a batch is expected to touch: tokens that each
    draw `sel` experts by a Zipf(1.1) popularity."""
    p = np.arange(1, c["experts"] + 1) ** -1.1
    p /= p.sum()
    lo, hi = 0.0, 1e6
    for _ in range(100):   # the scale at which `sel` experts are taken per token
        m = (lo + hi) / 2
        lo, hi = (m, hi) if np.sum(1 - np.exp(-m * p)) < c["sel"] else (lo, m)
    return float(np.sum(1 - np.exp(-lo * p * c["tokens"]))) if c["sel"] < c["experts"] else c["experts"]


def work(case):
    c, k = case, case["kind"]
    if k == "router":
        n, r = c["hidden"], c["rows"]
        return {"bytes": 4 * (r * n + 5 * n + r), "flops": 2 * r * n + 6 * n}
    if k in ("gemv", "head"):
        t = TYPES[c.get("type", "q6")]
        return {"bytes": wbytes(t, c["rows"], c["cols"]) + 4 * (c["cols"] + c["rows"]), "flops": 2 * c["rows"] * c["cols"]}
    if k == "qkv":
        return {"bytes": sum(wbytes(t, r, c["cols"]) + 4 * r for t, r in qkv_mats(c)) + 4 * c["cols"],
                "flops": sum(2 * r * c["cols"] for _, r in qkv_mats(c))}
    if k == "moe":
        S, n, f = c["sel"] + c["shared"], c["hidden"], c["ffn"]
        route = 4 * c["experts"] if c["route"] == "logits" else 8 * c["sel"]
        return {"bytes": c["layers"] * (S * expert_bytes(c) + 8 * n + route), "flops": c["layers"] * S * 6 * n * f}
    if k == "batch":
        S, n, f, T = c["sel"] + c["shared"], c["hidden"], c["ffn"], c["tokens"]
        return {"bytes": (distinct(c) + c["shared"]) * expert_bytes(c) + 8 * T * n + 4 * T * c["experts"],
                "flops": T * S * 6 * n * f}
    if k == "dense":
        n, qr, kr, f = c["hidden"], c["q_rows"], c["kv_rows"], c["ffn"]
        w = wbytes(Q4, qr + kr, n) + wbytes(Q6, kr, n) + wbytes(Q4, n, qr) + expert_bytes(c)
        return {"bytes": c["layers"] * (w + 4 * (qr + 2 * kr + 4 * n)),
                "flops": c["layers"] * 2 * ((qr + 2 * kr) * n + n * qr + 3 * n * f)}
    n, f = c["hidden"], c["ffn"]
    layer = c["sel"] * expert_bytes(c) + 4 * c["experts"] * n + 8 * n
    return {"bytes": c["layers"] * layer + wbytes(Q6, c["rows"], n) + 4 * c["rows"],
            "flops": c["layers"] * (c["sel"] * 6 * n * f + 2 * c["experts"] * n) + 2 * c["rows"] * n}


def tolerance(case):
    """fp32 sums of a row in any order were seen up to 2.4e-7 from 64 bits. A
    layer also quantizes a computed vector to 8 bits: a last-bit difference
    of it can move one quant by a step, which was seen as 2.5e-4 of that
    layer's output, and in a whole token as 1.3e-2 after 48 layers."""
    k = case["kind"]
    if k in ("router", "gemv", "qkv", "head"):
        return {"rel": 1e-6, "max": 1e-5}
    if k in ("moe", "batch"):
        return {"rel": 1e-3, "max": 2e-2}
    if k == "dense":
        return {"rel": 2e-3, "max": 5e-2}
    return {"rel": 3e-2, "max": 5e-1}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def dequant(t, w):
    """Blocks [..., nb, block bytes] to doubles [..., nb * 256]."""
    shape = w.shape[:-2] + (w.shape[-2] * 256,)
    b = w.reshape(-1, w.shape[-1])

    def f16(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    if t == Q4:
        s = b[:, 4:16].int()
        lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
        sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1).double() * f16(0)
        mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1).double() * f16(2)
        q = b[:, 16:144].reshape(-1, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32)
        return (sc[:, :, None] * q - mn[:, :, None]).reshape(shape)
    ql, qh = b[:, 0:128].reshape(-1, 2, 2, 32).int(), b[:, 128:192].reshape(-1, 2, 32).int()
    q = torch.stack([(ql[:, :, i & 1] >> (4 * (i >> 1)) & 15) | ((qh >> (2 * i) & 3) << 4) for i in range(4)], 2) - 32
    sc = b[:, 192:208].contiguous().view(torch.int8).double() * f16(208)
    return (sc[:, :, None] * q.reshape(-1, 16, 16)).reshape(shape)


def q8(x):
    """Rows of values as q8_1 blocks of 32 hold them (x rounded to fp32, each
    fp32 step of the block's definition rounded once)."""
    v = x.float().double().reshape(-1, 32)
    d = (v.abs().amax(1, keepdim=True) / 127.0).float().double()
    inv = torch.where(d > 0, 1.0 / d, torch.zeros_like(d)).float().double()
    p = (v * inv).float().double()
    return (torch.sign(p) * torch.floor(p.abs() + 0.5) * d.half().double()).reshape(x.shape)


def dot(t, w, x):
    """W . x for one row of x or several ([..., cols])."""
    rows = max(1, (1 << 28) // (w.shape[-2] * 256))
    return torch.cat([x @ dequant(t, w[i:i + rows]).T for i in range(0, w.shape[0], rows)], -1)


def ffn64(c, w, e, x):
    xq = q8(x)
    h = torch.nn.functional.silu(dot(Q4, w[0][e], xq)) * dot(Q4, w[1][e], xq)
    return dot(TYPES[c.get("down", "q6")], w[2][e], q8(h))


def norm64(x, w):
    return x / torch.sqrt((x * x).mean() + EPS) * w.double()


def moe64(c, w, lg, x):
    top, ids = torch.topk(lg.double(), c["sel"])
    return sum(p * ffn64(c, w, int(e), x) for p, e in zip(torch.softmax(top, -1), ids))


def exact(case, seed):
    c, k = case, case["kind"]
    v = inputs(c, seed)
    if k == "router":
        x = v["x"].double() + v["delta"].double()
        xn = norm64(x, v["norm"])
        y = v["w"].double() @ xn
        top, ids = torch.topk(y, c["sel"])
        return [x, xn, y, ids.to(torch.int32), torch.softmax(top, -1)]
    if k in ("gemv", "head"):
        x = v["x"].double() if c["act"] == "f32" else q8(v["x"])
        y = dot(TYPES[c.get("type", "q6")], v["w"], x)
        return [y, y.argmax().reshape(1)] if k == "head" else [y]
    if k == "qkv":
        x = v["x"].double() if c["act"] == "f32" else q8(v["x"])
        return [dot(t, w, x) for (t, _), w in zip(qkv_mats(c), v["w"])]
    if k == "moe":
        out = []
        for L in v["layers"]:
            y = moe64(c, L["w"], L["logits"], L["x"])
            out.append(y + ffn64(c, L["sh"], 0, L["x"]) if c["shared"] else y)
        return out
    if k == "batch":
        top, ids = torch.topk(v["logits"].double(), c["sel"], dim=-1)
        p = torch.softmax(top, -1)
        y = torch.zeros(c["tokens"], c["hidden"], device=DEV, dtype=torch.float64)
        for e in torch.unique(ids).tolist():
            t, r = torch.nonzero(ids == e, as_tuple=True)
            y[t] += p[t, r][:, None] * ffn64(c, v["w"], e, v["x"][t])
        return [y + ffn64(c, v["sh"], 0, v["x"]) if c["shared"] else y]
    if k == "dense":
        act = q8 if c["act"] == "dp4a" else (lambda z: z.float().double())
        x, out, ffn = v["x"].double(), [], None
        for L in v["layers"]:
            x = x if ffn is None else x + ffn
            xn = act(norm64(x, L["n1"]))
            qkv = [dot(t, w, xn) for (t, _), w in zip(qkv_mats(dict(c, cols=0)), L["qkv"])]
            att = dot(Q4, L["o"], act(qkv[0]))
            x = x + att
            ffn = ffn64(c, L["ffn"], 0, norm64(x, L["n2"]))
            out += qkv + [att, ffn]
        return out
    x, y = v["x"].double(), None
    for L in v["layers"]:
        x = x if y is None else x + y
        xn = norm64(x, L["norm"]).float().double()
        y = moe64(c, L["w"], L["router"].double() @ xn, xn)
    lg = dot(Q6, v["head"], q8(norm64(x + y, v["norm"])))
    return [y, lg, lg.argmax().reshape(1)]
