"""The work that a user of this library has it do, as cases to be timed.

The two models behind the entry points set the shapes: a mixture-of-experts model in Q4_0 (hidden 2816, 128 experts of
704, 8 a token, a shared FFN of 2112 beside them, a Q6_K head over 262144 tokens; and the benchmark's own 2048 x 768
layer) and a dense model in Q4_K and Q6_K (hidden 4096, FFN 12288) that decodes on int8 activations, verifies a few
drafted tokens at a time and takes its prompts through the prefill GEMMs.

A case is a dict with a "kind" (one chain of public operator calls each, see the `_prepare_*` / `_run_*` pairs) and sizes.
"""
import math

import torch

from leviathan_amd import capi, ops

KINDS = ("gemv", "shared_ffn", "moe", "decode", "head", "verify", "q8_ffn", "prefill")


def listed():
    return [
        # One Q4_0 decode GEMV called by itself, as a program that mixes its own operators with the library's does:
        # the smallest call, 9.5 MB.
        {"name": "gemv 4096x4096", "kind": "gemv", "in_dim": 4096, "rows": 4096},
        # The shared expert of one decoded token: six dependent operators of a few megabytes.
        {"name": "shared ffn 2816/2112", "kind": "shared_ffn", "hidden": 2816, "inter": 2112},
        # One token through the MoE block of eight successive layers, each with its own router and experts.
        {"name": "moe 1 token x8 layers", "kind": "moe", "hidden": 2048, "inter": 768, "experts": 128, "top_k": 8,
         "tokens": 1, "layers": 8},
        # One token through four whole FFN blocks, recorded once and replayed, as a decode loop does.
        {"name": "decode program 4 layers", "kind": "decode", "hidden": 2816, "inter": 704, "shared": 2112,
         "experts": 128, "top_k": 8, "layers": 4},
        # A batch of 64 sequences decoding together.
        {"name": "moe 64 tokens", "kind": "moe", "hidden": 2048, "inter": 768, "experts": 128, "top_k": 8,
         "tokens": 64, "layers": 1},
        # The MoE block over a prompt of ordinary, ragged length.
        {"name": "moe prompt 1000", "kind": "moe", "hidden": 2816, "inter": 704, "experts": 128, "top_k": 8,
         "tokens": 1000, "layers": 1},
        # The greedy token from the full vocabulary.
        {"name": "head 262144x2816", "kind": "head", "in_dim": 2816, "rows": 262144, "ncol": 1, "greedy": True},
        # Four drafted tokens verified in one read of an up projection, RMSNorm in front.
        {"name": "verify 4 12288x4096", "kind": "verify", "in_dim": 4096, "rows": 12288, "ncol": 4},
        # One token through a dense FFN on int8 activations (decode), and five (verify).
        {"name": "q8 ffn 4096/12288 n1", "kind": "q8_ffn", "hidden": 4096, "inter": 12288, "ncol": 1},
        {"name": "q8 ffn 4096/12288 n5", "kind": "q8_ffn", "hidden": 4096, "inter": 12288, "ncol": 5},
        # A full prefill chunk through the up projection, and a short prompt through a Q6_K down projection.
        {"name": "prefill q4_k 512", "kind": "prefill", "fmt": "q4_k", "in_dim": 4096, "rows": 12288, "tokens": 512},
        {"name": "prefill q6_k 77", "kind": "prefill", "fmt": "q6_k", "in_dim": 12288, "rows": 4096, "tokens": 77},
    ]


# ---- sizes ---------------------------------------------------------------------------------------------------------

def _log(rng, low, high, step=1):
    """A multiple of `step` between low and high, its logarithm uniform."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return min(high // step, max(-(-low // step), round(v / step))) * step


def _draw(rng):
    kind = rng.choice(KINDS)
    c = {"kind": kind}
    if kind == "gemv":                       # any projection of a decoded token, an expert's slice among them
        c.update(in_dim=_log(rng, 256, 16384, 32), rows=_log(rng, 700, 40000))
    elif kind == "shared_ffn":
        c.update(hidden=_log(rng, 1024, 5120, 64), inter=_log(rng, 512, 6144, 64))
    elif kind in ("moe", "decode"):
        c.update(hidden=_log(rng, 1024, 4096, 128), inter=_log(rng, 256, 1536, 64), experts=rng.choice((32, 60, 64, 128, 256)),
                 top_k=rng.choice((2, 4, 6, 8)))
        if kind == "moe":                    # one sequence, a batch of them, a prompt
            c.update(tokens=_log(rng, 1, 1000), layers=1)
        else:
            c.update(shared=_log(rng, 512, 4096, 64), layers=rng.choice((1, 2, 3, 4)))
    elif kind == "head":
        c.update(in_dim=_log(rng, 1024, 6144, 256), rows=_log(rng, 16000, 262144), ncol=rng.choice((1, 1, 2, 3, 4, 8)))
        c["greedy"] = c["ncol"] == 1
    elif kind == "verify":                   # up, down and attention projections
        c.update(in_dim=_log(rng, 1024, 12288, 256), rows=_log(rng, 1000, 16384), ncol=rng.randint(1, 8))
    elif kind == "q8_ffn":
        c.update(hidden=_log(rng, 1024, 6144, 256), inter=_log(rng, 2048, 16384, 256), ncol=rng.choice((1, 1, 2, 3, 4, 5, 8, 16)))
    else:
        c.update(fmt=rng.choice(("q4_k", "q6_k")), in_dim=_log(rng, 1024, 12288, 256), rows=_log(rng, 1000, 32000),
                 tokens=_log(rng, 17, 1024))
    return c


def draw(rng):
    listed_work = [work(c) for c in listed()]
    most_bytes, most_flops = (max(w[k] for w in listed_work) for k in ("bytes", "flops"))
    while True:
        c = _draw(rng)
        w = work(c)
        if w["bytes"] <= most_bytes and w["flops"] <= most_flops:
            return c


# ---- weights and activations -----------------------------------------------------------------------------------------

_CTX = []


def _ctx():
    """The one context of the program, on a stream of its own (recording needs one)."""
    if not _CTX:
        _CTX.append(ops.Context(0, own_stream=True))
    return _CTX[0]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _bytes(g, *shape):
    n = math.prod(shape)
    return torch.empty(-(-n // 8), dtype=torch.int64, device="cuda").random_(-2**63, 2**63 - 1, generator=g).view(torch.uint8)[:n].reshape(shape)


def _half(g, n, sigma):
    """n scales |N(0, sigma)| in fp16, as bytes."""
    return (torch.randn(n, 1, device="cuda", generator=g) * sigma).abs().half().view(torch.uint8)


def _q4_0(g, rows, in_dim):
    """Uniform 4-bit codes, weights of about unit gain: 4.6 d is their standard deviation."""
    n = rows * in_dim // 32
    w = _bytes(g, n, 18)
    w[:, 0:2] = _half(g, n, 1 / (4.6 * math.sqrt(in_dim)))
    return w.reshape(-1)


def _q4_k(g, rows, in_dim):
    n = rows * in_dim // 256
    w = _bytes(g, n, 144)                    # 6-bit scales and mins and the codes: uniform
    w[:, 0:2] = _half(g, n, 1 / (170 * math.sqrt(in_dim)))
    w[:, 2:4] = _half(g, n, 1 / (25 * math.sqrt(in_dim)))
    return w.reshape(-1)


def _q6_k(g, rows, in_dim):
    n = rows * in_dim // 256
    w = _bytes(g, n, 210)
    w[:, 192:208] = torch.randint(-32, 32, (n, 16), device="cuda", generator=g, dtype=torch.int8).view(torch.uint8)
    w[:, 208:210] = _half(g, n, 1 / (340 * math.sqrt(in_dim)))
    return w.reshape(-1)


def _normal(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def _gain(g, n):
    return 1 + 0.1 * _normal(g, n)


def _f32(*shape):
    return torch.empty(shape, dtype=torch.float32, device="cuda")


def _moe_weights(g, c):
    h, i, e = c["hidden"], c["inter"], c["experts"]
    pool = torch.cat([_q4_0(g, e * i, h), _q4_0(g, e * i, h), _q4_0(g, e * h, i)])
    gu = e * i * (h // 32) * 18
    return {"pools": ops.Context.moe_pools(pool, h, i, e, 0, gu, 2 * gu), "router": 0.02 * _normal(g, e, h)}


def _moe_out(c):
    t, k = c.get("tokens", 1), c["top_k"]
    return {"y": _f32(t, c["hidden"]), "ids": torch.empty((t, k), dtype=torch.int32, device="cuda"), "weights": _f32(t, k)}


def _ffn_weights(g, h, i):
    return {"norm": _gain(g, h), "gate": _q4_0(g, i, h), "up": _q4_0(g, i, h), "down": _q4_0(g, h, i), "post": _gain(g, h),
            "bufs": (_f32(h), _f32(2 * i), _f32(i), _f32(h))}


# ---- one pass of each kind -------------------------------------------------------------------------------------------

def _prepare_gemv(c, g):
    return {"w": _q4_0(g, c["rows"], c["in_dim"]), "x": _normal(g, c["in_dim"]), "y": _f32(c["rows"])}


def _run_gemv(s, c, ctx):
    return ctx.q4_0_gemv(s["w"], s["x"], c["in_dim"], c["rows"], y=s["y"])


def _prepare_shared_ffn(c, g):
    return dict(_ffn_weights(g, c["hidden"], c["inter"]), x=_normal(g, c["hidden"]))


def _run_shared_ffn(s, c, ctx):
    return ctx.shared_expert_ffn(s["x"], s["norm"], s["gate"], s["up"], s["down"], s["post"], c["hidden"], c["inter"], bufs=s["bufs"])


def _prepare_moe(c, g):
    return {"layers": [dict(_moe_weights(g, c), x=_normal(g, c["tokens"], c["hidden"]), **_moe_out(c)) for _ in range(c["layers"])]}


def _run_moe(s, c, ctx):
    return [ctx.moe_layer_q4_0(m["pools"], m["router"], m["x"], c["top_k"], c["tokens"], y=m["y"], ids=m["ids"], weights=m["weights"])
            for m in s["layers"]]


def _decode_step(s, c, ctx):
    """x of a layer is the sum of the layer before it: the residual, the shared FFN and the routed experts on the
    normalised residual. Every layer's x is a buffer of its own, so a replay finds its input as it was."""
    x = s["x"]
    for m in s["layers"]:
        h, shared = ctx.shared_expert_ffn(x, m["norm"], m["gate"], m["up"], m["down"], m["post"], c["hidden"], c["shared"], bufs=m["bufs"])
        ctx.moe_layer_q4_0(m["pools"], m["router"], h[None], c["top_k"], 1, y=m["y"], ids=m["ids"], weights=m["weights"])
        ctx.rmsnorm(m["y"], c["hidden"], 1, weight=m["post"], y=m["out"])
        ctx.axpy(shared, m["out"], 1.0, c["hidden"])
        ctx.axpy(x, m["out"], 1.0, c["hidden"])
        x = m["out"]
    return x


def _prepare_decode(c, g):
    s = {"x": _normal(g, c["hidden"])}
    s["layers"] = [dict(_moe_weights(g, c), **_ffn_weights(g, c["hidden"], c["shared"]), **_moe_out(c), out=_f32(c["hidden"]))
                   for _ in range(c["layers"])]
    ctx = _ctx()
    torch.cuda.synchronize()
    _decode_step(s, c, ctx)                  # grows the context's scratch: recording may not
    ctx.sync()
    ctx.program_begin()
    _decode_step(s, c, ctx)
    s["program"] = ctx.program_end()
    return s


def _run_decode(s, c, ctx):
    s["program"].run()
    return [(m["out"], m["ids"], m["weights"]) for m in s["layers"]]


def _prepare_head(c, g):
    return {"w": _q6_k(g, c["rows"], c["in_dim"]), "x": _normal(g, c["ncol"], c["in_dim"]), "gain": _gain(g, c["in_dim"]),
            "y": _f32(c["ncol"], c["rows"])}


def _run_head(s, c, ctx):
    if c["greedy"]:
        return ctx.q6_k_gemv(s["w"], s["x"], c["in_dim"], c["rows"], y=s["y"], argmax=True)
    y = ctx.q6_k_gemv_ncol(s["w"], s["x"], c["in_dim"], c["rows"], c["ncol"], gain=s["gain"], y=s["y"])
    return (y,) + ctx.argmax(y, c["rows"], c["ncol"])


def _prepare_verify(c, g):
    return {"w": _q4_k(g, c["rows"], c["in_dim"]), "x": _normal(g, c["ncol"], c["in_dim"]), "gain": _gain(g, c["in_dim"]),
            "y": _f32(c["ncol"], c["rows"])}


def _run_verify(s, c, ctx):
    return ctx.q4_k_gemv_ncol(s["w"], s["x"], c["in_dim"], c["rows"], c["ncol"], gain=s["gain"], y=s["y"])


def _prepare_q8_ffn(c, g):
    h, i, n = c["hidden"], c["inter"], c["ncol"]
    return {"gate": _q4_k(g, i, h), "up": _q4_k(g, i, h), "down": _q6_k(g, h, i), "gain": _gain(g, h), "x": _normal(g, n, h),
            "g": _f32(n, i), "u": _f32(n, i), "y": _f32(n, h)}


def _run_q8_ffn(s, c, ctx):
    h, i, n = c["hidden"], c["inter"], c["ncol"]
    xq, xs = ctx.norm_quant_q8(s["x"], h, n, gain=s["gain"])
    gate = ctx.q4_k_gemv_q8(s["gate"], xq, xs, h, i, n, y=s["g"])
    up = ctx.q4_k_gemv_q8(s["up"], xq, xs, h, i, n, y=s["u"])
    aq, as_ = ctx.swiglu_quant_q8(gate, up)
    return gate, up, ctx.q6_k_gemv_q8(s["down"], aq, as_, i, h, n, y=s["y"])


def _prepare_prefill(c, g):
    make = _q4_k if c["fmt"] == "q4_k" else _q6_k
    return {"w": make(g, c["rows"], c["in_dim"]), "x": _normal(g, c["tokens"], c["in_dim"]).half(), "y": _f32(c["tokens"], c["rows"])}


def _run_prefill(s, c, ctx):
    gemm = ctx.q4_k_gemm_prefill if c["fmt"] == "q4_k" else ctx.q6_k_gemm_prefill
    return gemm(s["w"], s["x"], c["in_dim"], c["rows"], c["tokens"], y=s["y"])


def prepare(case, seed):
    state = globals()["_prepare_" + case["kind"]](case, _gen(seed))
    state.update(case=case, ctx=_ctx(), run=globals()["_run_" + case["kind"]])
    torch.cuda.synchronize()                 # inputs are made on torch's stream, the library works on its own
    return state


def run(state):
    return state["run"](state, state["case"], state["ctx"])


# ---- what a pass cannot do without -------------------------------------------------------------------------------------

def _expert_bytes(c):
    """Gate, up and down of the experts that `tokens` tokens reach, each read once, and the router."""
    t, e, k = c.get("tokens", 1), c["experts"], c["top_k"]
    reached = e * (1 - (1 - k / e) ** t)
    return reached * 3 * c["hidden"] * c["inter"] * 18 / 32 + 4 * e * c["hidden"]


def _moe_flops(c):
    return 2 * c.get("tokens", 1) * (c["top_k"] * 3 * c["hidden"] * c["inter"] + c["experts"] * c["hidden"])


def work(case):
    c, kind = case, case["kind"]
    if kind == "gemv":
        w, act, flops = c["rows"] * c["in_dim"] * 18 / 32, c["in_dim"] + c["rows"], 2 * c["rows"] * c["in_dim"]
    elif kind == "shared_ffn":
        w, act, flops = 3 * c["hidden"] * c["inter"] * 18 / 32, 5 * c["hidden"], 6 * c["hidden"] * c["inter"]
    elif kind == "moe":
        n = c["layers"]
        w, act, flops = n * _expert_bytes(c), n * c["tokens"] * (2 * c["hidden"] + 2 * c["top_k"]), n * _moe_flops(c)
    elif kind == "decode":
        n = c["layers"]
        w = n * (_expert_bytes(c) + 3 * c["hidden"] * c["shared"] * 18 / 32)
        act, flops = n * 4 * c["hidden"], n * (_moe_flops(c) + 6 * c["hidden"] * c["shared"])
    elif kind == "q8_ffn":
        w = c["hidden"] * c["inter"] * (2 * 144 + 210) / 256
        act, flops = c["ncol"] * (2 * c["hidden"] + 2 * c["inter"]), 6 * c["ncol"] * c["hidden"] * c["inter"]
    elif kind in ("head", "verify"):
        w = c["rows"] * c["in_dim"] * (210 if kind == "head" else 144) / 256
        act, flops = c["ncol"] * (c["in_dim"] + c["rows"]), 2 * c["ncol"] * c["rows"] * c["in_dim"]
    else:
        w = c["rows"] * c["in_dim"] * (144 if c["fmt"] == "q4_k" else 210) / 256
        act, flops = c["tokens"] * (c["in_dim"] / 2 + c["rows"]), 2 * c["tokens"] * c["rows"] * c["in_dim"]
    return {"bytes": w + 4 * act, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "prefill":                    # weights rounded to fp16 (unit roundoff 2^-11), f32 sums
        return {"rel": 5e-4}
    if kind == "q8_ffn":                     # an activation at the border of two int8 codes may take either
        return {"rel": 1e-3}
    if kind == "decode":                     # f32 rounding, carried through the layers; scores that tie in f32
        return {"rel": 1e-4, "differ": 0.002}
    if kind in ("moe", "head"):              # f32 sums; scores (logits) that tie in f32
        return {"rel": 1e-5, "differ": 0.002}
    return {"rel": 1e-5}
