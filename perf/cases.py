"""What the ternary backend is timed on: its linear layers, FFN and MoE block from one token to a full prompt, and the
quantiser, each through the entry points of ferrisres_amd.Context.

Widths are those of the benchmark and the tests: 2048 x 2048 (the reference's single linear), hidden 2048 / inner 5632,
4096 / 11008 and 5120 / 13824. Calls of up to 16 tokens, which a serving loop issues again for each token, are
captured once into a graph and replayed (all but the single linear, which is called as it is); longer ones are
plain calls.
"""
from __future__ import annotations

import math

import torch

import ferrisres_amd as frx

DEV = "cuda:0"
DT = {"f32": torch.float32, "bf16": torch.bfloat16}
PAIRS = ((0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3))  # the two kept positions of a 2:4 group, by pattern
MOST_MACS = 2048 * 4096 * 11008
_ctx = None


def listed():
    return [
        # one token through the reference's single linear, f32 in and out, called by itself: latency
        {"name": "linear_1tok_f32", "kind": "linear", "m": 1, "k": 2048, "n": 2048, "dtype": "f32", "out": "f32",
         "bias": False, "graph": False},
        # a decode step of one sequence: q/k/v on one x, o, FFN, over four layers of a 7B model
        {"name": "layers_1tok_bf16", "kind": "layers", "m": 1, "h": 4096, "i": 11008, "layers": 4, "dtype": "bf16",
         "graph": True},
        # the same step for a full decode batch
        {"name": "layers_16tok_bf16", "kind": "layers", "m": 16, "h": 4096, "i": 11008, "layers": 2, "dtype": "bf16",
         "graph": True},
        # a small batch on a small model in f32, the reference's own activation type
        {"name": "layers_5tok_f32", "kind": "layers", "m": 5, "h": 2048, "i": 5632, "layers": 4, "dtype": "f32",
         "graph": True},
        # a chunk of a prompt through the FFN, an odd number of tokens
        {"name": "ffn_333tok_bf16", "kind": "ffn", "m": 333, "h": 4096, "i": 11008, "dtype": "bf16", "act": "silu",
         "graph": False},
        # prompt processing: the widest linear of a 7B model over 2048 tokens
        {"name": "linear_2048tok_bf16", "kind": "linear", "m": 2048, "k": 4096, "n": 11008, "dtype": "bf16",
         "out": "bf16", "bias": False, "graph": False},
        # prompt processing in f32 in and out (the drop-in of the reference's dispatch), 13B width, odd token count
        {"name": "linear_517tok_f32", "kind": "linear", "m": 517, "k": 5120, "n": 13824, "dtype": "f32", "out": "f32",
         "bias": True, "graph": False},
        # 2:4 weights: a small f32 decode batch over the reference's metadata, and a prompt over resident weights
        {"name": "sp24_8tok_f32", "kind": "sp24", "m": 8, "k": 4096, "n": 11008, "dtype": "f32", "out": "f32",
         "prepared": False, "graph": True},
        {"name": "sp24_2048tok_bf16", "kind": "sp24", "m": 2048, "k": 4096, "n": 11008, "dtype": "bf16", "out": "bf16",
         "prepared": True, "graph": False},
        # the MoE block: a decode batch, and a prompt chunk
        {"name": "moe_8tok_bf16", "kind": "moe", "m": 8, "h": 2048, "i": 5632, "e": 16, "top_k": 2, "dtype": "bf16",
         "act": "silu", "graph": True},
        {"name": "moe_512tok_bf16", "kind": "moe", "m": 512, "h": 2048, "i": 5632, "e": 16, "top_k": 2,
         "dtype": "bf16", "act": "silu", "graph": False},
        # re-quantising a layer's shadow weights after an optimiser step
        {"name": "quantize_f32", "kind": "quantize", "n": 11008, "k": 4096, "dtype": "f32", "rule": "absmean"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, step):
    return max(step, _log_int(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(("linear", "linear", "layers", "ffn", "sp24", "moe", "quantize"))
    dtype = rng.choice(("bf16", "bf16", "f32"))
    halves = 2 if dtype == "f32" else 1
    if kind == "quantize":
        while True:
            n, k = _log_int(rng, 512, 16384), _width(rng, 1024, 14336, 16 if rng.random() < 0.3 else 256)
            if n * k <= 11008 * 4096:
                return {"kind": kind, "n": n, "k": k, "dtype": dtype, "rule": rng.choice(("absmean", "ste"))}
    if kind in ("linear", "sp24"):
        ragged = rng.random() < 0.25  # widths that are no multiples of 64
        m = _log_int(rng, 1, 2048)
        while True:
            k, n = _width(rng, 1024, 14336, 16 if ragged else 64), _width(rng, 1024, 14336, 4 if ragged else 64)
            if m * k * n * halves <= MOST_MACS:
                break
        c = {"kind": kind, "m": m, "k": k, "n": n, "dtype": dtype, "out": rng.choice((dtype, "f32")),
             "graph": m <= 16}
        if kind == "linear":
            c["bias"] = rng.random() < 0.25
        else:
            c["prepared"] = dtype == "bf16" and k % 64 == 0 and rng.random() < 0.5
        return c
    if kind == "moe":
        while True:
            h, i, e = _width(rng, 1024, 4096, 64), _width(rng, 1024, 8192, 64), rng.choice((8, 16, 32))
            m, top_k = _log_int(rng, 1, 512), rng.choice((1, 2, 2, 4))
            if h * i * e <= 2048 * 5632 * 16 and m * top_k * h * i * halves <= 1024 * 2048 * 5632:
                return {"kind": kind, "m": m, "h": h, "i": i, "e": e, "top_k": top_k, "dtype": dtype,
                        "act": rng.choice(("silu", "gelu")), "graph": m <= 16}
    h, i = _width(rng, 1024, 5120, 64), _width(rng, 2048, 13824, 64)
    if kind == "layers":
        return {"kind": kind, "m": _log_int(rng, 1, 16), "h": h, "i": i, "layers": 2, "dtype": dtype, "graph": True}
    return {"kind": kind, "m": _log_int(rng, 1, 680 // halves), "h": h, "i": i, "dtype": dtype,
            "act": rng.choice(("silu", "gelu")), "graph": False}


# ---- inputs, all from the seed --------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _ternary(g, n, k):
    """Codes of an absmean-quantised normal matrix (38% zeros), packed [n][k/16]."""
    c = torch.randn((n, k // 16, 16), generator=g, device=DEV).round_().clamp_(-1, 1).to(torch.int32).add_(1)
    sh = torch.arange(0, 32, 2, device=DEV, dtype=torch.int32)
    return torch.sum(c << sh, dim=2, dtype=torch.int32)


def _sparse24(g, n, k):
    """2:4 metadata [n][ceil(ceil(k/4)/6)]: six 5-bit groups (pattern, two sign bits) per word."""
    groups = k // 4
    words = (groups + 5) // 6
    v = torch.randint(0, 6, (n, words * 6), generator=g, device=DEV, dtype=torch.int32)
    v += torch.randint(0, 4, (n, words * 6), generator=g, device=DEV, dtype=torch.int32) << 3
    v[:, groups:] = 0
    sh = torch.arange(0, 30, 5, device=DEV, dtype=torch.int32)
    return torch.sum(v.view(n, words, 6) << sh, dim=2, dtype=torch.int32)


def _scales(g, n):
    return 0.016 + 0.008 * torch.rand((n,), generator=g, device=DEV)


def _acts(g, m, k, dtype):
    """Normalised activations: channels of uneven gain, a few of them far larger than the rest."""
    gain = torch.exp(0.3 * torch.randn((k,), generator=g, device=DEV))
    gain *= torch.where(torch.rand((k,), generator=g, device=DEV) < 1 / 256, 12.0, 1.0)
    return (torch.randn((m, k), generator=g, device=DEV) * gain).to(DT[dtype]).contiguous()


def _inputs(c, seed):
    """The state's tensors: activations, weights and scales."""
    g = _gen(seed)
    kind = c["kind"]
    if kind == "quantize":
        return {"w": (0.02 * torch.randn((c["n"], c["k"]), generator=g, device=DEV)).to(DT[c["dtype"]])}
    if kind in ("linear", "sp24"):
        n, k = c["n"], c["k"]
        t = {"x": _acts(g, c["m"], k, c["dtype"]), "w": (_ternary if kind == "linear" else _sparse24)(g, n, k),
             "s": _scales(g, n)}
        if c.get("bias"):
            t["bias"] = 0.1 * torch.randn((n,), generator=g, device=DEV)
        return t
    h, i, m = c["h"], c["i"], c["m"]
    mat = lambda n, k: (_ternary(g, n, k), _scales(g, n))  # noqa: E731
    if kind == "layers":
        return [{"x": _acts(g, m, h, c["dtype"]), "a": _acts(g, m, h, c["dtype"]), "f": _acts(g, m, h, c["dtype"]),
                 "q": mat(h, h), "k": mat(h, h), "v": mat(h, h), "o": mat(h, h),
                 "gate": mat(i, h), "up": mat(i, h), "down": mat(h, i)} for _ in range(c["layers"])]
    t = {"x": _acts(g, m, h, c["dtype"])}
    if kind == "moe":
        t["router"] = (torch.randn((c["e"], h), generator=g, device=DEV) / math.sqrt(h)).to(DT[c["dtype"]])
    count = c["e"] if kind == "moe" else 1
    for name, n, k in (("gate", i, h), ("up", i, h), ("down", h, i)):
        t[name] = [mat(n, k) for _ in range(count)]
    return t


def _context():
    global _ctx
    if _ctx is None:
        _ctx = frx.Context(0)
    return _ctx


ACT = {"silu": frx.ACT_SILU, "gelu": frx.ACT_GELU_TANH}
RULE = {"absmean": frx.QUANT_ABSMEAN, "ste": frx.QUANT_STE}


def _call(c, ctx, t, out):
    """The entry points of one pass, in order, into the tensors of `out`."""
    kind = c["kind"]
    if kind == "linear":
        ctx.ternary_linear(t["w"], t["s"], t["x"], out["y"], bias=t.get("bias"))
    elif kind == "sp24":
        if c["prepared"]:
            ctx.sparse24_prepared_linear(t["prepared"], t["s"], t["x"], out["y"])
        else:
            ctx.sparse24_ternary_linear(t["w"], t["s"], t["x"], out["y"])
    elif kind == "layers":
        for lt, lo in zip(t, out):
            qkv = (lt["q"], lt["k"], lt["v"])
            ctx.ternary_linear_group(lt["x"], [w for w, _ in qkv], [s for _, s in qkv], [lo["q"], lo["k"], lo["v"]])
            ctx.ternary_linear(*lt["o"], lt["a"], lo["o"])
            ctx.ternary_ffn(lt["f"], *lt["gate"], *lt["up"], *lt["down"], lo["f"])
    elif kind == "ffn":
        ctx.ternary_ffn(t["x"], *t["gate"][0], *t["up"][0], *t["down"][0], out["y"], act=ACT[c["act"]])
    elif kind == "moe":
        ws = [[w[p] for w in t[name]] for name in ("gate", "up", "down") for p in (0, 1)]
        ctx.moe_ternary_ffn(t["x"], t["router"], *ws, out["y"], top_k=c["top_k"], act=ACT[c["act"]],
                            topk_idx=out["idx"], topk_w=out["weight"])
    else:
        ctx.quantize_ternary(t["w"], RULE[c["rule"]], out["packed"], out["scale"])


def prepare(case, seed):
    ctx = _context()
    t = _inputs(case, seed)
    kind = case["kind"]
    new = lambda *shape, dtype=torch.float32: torch.zeros(shape, dtype=dtype, device=DEV)  # noqa: E731
    if kind == "quantize":
        out = {"packed": new(case["n"], case["k"] // 16, dtype=torch.int32), "scale": new(case["n"])}
    elif kind in ("linear", "sp24"):
        out = {"y": new(case["m"], case["n"], dtype=DT[case["out"]])}
    elif kind == "layers":
        out = [{n: new(case["m"], case["h"], dtype=DT[case["dtype"]]) for n in "qkvof"} for _ in t]
    else:
        out = {"y": new(case["m"], case["h"], dtype=torch.float32 if kind == "moe" else DT[case["dtype"]])}
    if kind == "moe":
        out["idx"] = new(case["m"], case["top_k"], dtype=torch.int32)
        out["weight"] = new(case["m"], case["top_k"])
    if case.get("prepared"):
        t["prepared"] = new(case["n"], case["k"] // 16, dtype=torch.int32)
        ctx.sparse24_prepare(t["w"], case["k"], t["prepared"])
    state = {"case": case, "ctx": ctx, "in": t, "out": out, "graph": None}
    if case.get("graph"):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        ctx.set_stream(side)
        with torch.cuda.stream(side):
            _call(case, ctx, t, out)  # the context's workspaces grow outside the capture
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            _call(case, ctx, t, out)
        ctx.set_stream(torch.cuda.current_stream())
        state["graph"] = graph
    return state


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        _call(state["case"], state["ctx"], state["in"], state["out"])
    return state["out"]


# ---- what a pass has to move and to compute -------------------------------------------------------------------------

def _expected_experts(c):
    """Experts that at least one of the tokens reaches when each takes top_k of e at random."""
    return c["e"] * (1 - (1 - c["top_k"] / c["e"]) ** c["m"])


def work(case):
    kind = case["kind"]
    width = 2 if case["dtype"] == "bf16" else 4
    if kind == "quantize":
        n, k = case["n"], case["k"]
        return {"bytes": n * k * width + n * k / 4 + 4 * n, "flops": 2 * n * k}
    m = case["m"]
    if kind in ("linear", "sp24"):
        n, k = case["n"], case["k"]
        per_row = 4 * ((k // 4 + 5) // 6) if kind == "sp24" else k / 4
        if case.get("prepared"):
            per_row = k / 4
        out = 2 if case["out"] == "bf16" else 4
        # a 2:4 matrix has half of its products left
        return {"bytes": n * (per_row + 4) + m * k * width + m * n * out,
                "flops": 2 * m * n * k // (2 if kind == "sp24" else 1)}
    h, i = case["h"], case["i"]
    ffn = 3 * h * i / 4 + 4 * (2 * i + h)
    if kind == "layers":
        return {"bytes": case["layers"] * (ffn + 4 * (h * h / 4 + 4 * h) + 8 * m * h * width),
                "flops": case["layers"] * 2 * m * (4 * h * h + 3 * h * i)}
    if kind == "ffn":
        return {"bytes": ffn + 2 * m * h * width, "flops": 6 * m * h * i}
    return {"bytes": _expected_experts(case) * ffn + case["e"] * h * width + m * h * (width + 4) + m * case["top_k"] * 8,
            "flops": 2 * m * h * case["e"] + 6 * m * case["top_k"] * h * i}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"  # codes and scales are the reference's, its order of additions included
    out = case.get("out") or ("f32" if kind == "moe" else case["dtype"])
    if out == "bf16":
        return {"rel": 7e-3}  # one rounding to 8 bits of each output: 1.7e-3 off the exact ones
    # f32 activations travel as pairs of bf16, 2.5e-6 off the exact outputs; inner activations do so too, 5e-6
    return {"rel": 1e-5 if kind in ("linear", "sp24") else 2e-5}


# ---- the same outputs in 64 bits -------------------------------------------------------------------------------------

def _dense64(w):
    n, words = w.shape
    sh = torch.arange(0, 32, 2, device=w.device, dtype=torch.int32)
    return (((w[:, :, None] >> sh) & 3) - 1).view(n, words * 16).double()


def _sparse64(w, k):
    n, words = w.shape
    sh = torch.arange(0, 30, 5, device=w.device, dtype=torch.int32)
    v = ((w[:, :, None] >> sh) & 31).view(n, words * 6)[:, :k // 4]
    pairs = torch.tensor(PAIRS, device=w.device)[(v & 7).long()]
    full = torch.zeros((n, k // 4, 4), dtype=torch.float64, device=w.device)
    for j in range(2):
        full.scatter_(2, pairs[:, :, j:j + 1], (1 - 2 * ((v >> (3 + j)) & 1)).double()[:, :, None])
    return full.view(n, k)


def _linear64(x, mat):
    return (x.double() @ _dense64(mat[0]).t()) * mat[1].double()


def _ffn64(x, gate, up, down, act):
    g = _linear64(x, gate)
    g = torch.nn.functional.silu(g) if act == "silu" else torch.nn.functional.gelu(g, approximate="tanh")
    return _linear64(g * _linear64(x, up), down)


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "quantize":
        alpha = t["w"].double().abs().mean(dim=1)
        return {"packed": None, "scale": alpha / 0.7978845608 if case["rule"] == "absmean" else alpha}
    if kind == "linear":
        y = _linear64(t["x"], (t["w"], t["s"]))
        return {"y": y + t["bias"].double() if "bias" in t else y}
    if kind == "sp24":
        return {"y": (t["x"].double() @ _sparse64(t["w"], case["k"]).t()) * t["s"].double()}
    if kind == "layers":
        return [{**{n: _linear64(lt["x"], lt[n]) for n in "qkv"}, "o": _linear64(lt["a"], lt["o"]),
                 "f": _ffn64(lt["f"], lt["gate"], lt["up"], lt["down"], "silu")} for lt in t]
    if kind == "ffn":
        return {"y": _ffn64(t["x"], t["gate"][0], t["up"][0], t["down"][0], case["act"])}
    p = torch.softmax(t["x"].double() @ t["router"].double().t(), dim=1)
    weight, idx = torch.sort(p, dim=1, descending=True, stable=True)
    weight, idx = weight[:, :case["top_k"]], idx[:, :case["top_k"]]
    weight = weight / weight.sum(dim=1, keepdim=True)
    y = torch.zeros(t["x"].shape, dtype=torch.float64, device=DEV)
    for e in range(case["e"]):
        rows, slot = torch.nonzero(idx == e, as_tuple=True)
        if len(rows):
            y[rows] += weight[rows, slot, None] * _ffn64(t["x"][rows], t["gate"][e], t["up"][e], t["down"][e],
                                                         case["act"])
    return {"y": y, "idx": None, "weight": weight}
