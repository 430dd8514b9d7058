"""The calls that a user of the MoE layer library makes, for timing and comparing two builds.

Every case is one pass through the public Python binding (mimoe) over synthetic
layers of the shapes the library is made for:

  moondream3      D 2048, 64 experts, top-8, inner 1024, fused [h | g] tables, LayerNorm
  qwen3omni       D 2048, 128 experts, top-8, inner 768, gate and up tables, RMSNorm
  diffusiongemma  D 2816, 128 experts, top-8, inner 704, router on its own rows,
                  softmax over all experts, per-expert scale
  nemotronomni    128 experts, top-6, inner 1856, relu^2 without a gate, sigmoid
                  router with a selection bias, shared expert of 3712 (width 2688)

in the table types the GGUF files carry: Q4_K with a Q4_K or Q6_K down table, Q6_K
throughout, and the converters' Q8_0, Q5_0, Q4_0 and F16.

A case's plain values: `model`, `op` (forward | norm | own_router | caller_ids), `T`
tokens, `layers` (each on its own rows, one call after the other, as the MoE blocks of
one step), `gate` / `down` table types, `act`, `tiled` (the layer carries the load-time
tiled copies), `zipf` (skewed router bias with 16 idle experts), `routing` (the caller
asks for the routing outputs).

Weights are N(0, 0.02) quantized here, in torch, with the formats' plain
round-to-nearest quantizers: `exact` then has the tables' values in float64 without the
library's code.
"""
import ctypes
import math
import pathlib
import sys

import torch

sys.path.insert(0, str(pathlib.Path.cwd() / "skyvision.cpp_amd"))

import mimoe as M  # noqa: E402

F64 = torch.float64
TYPES = {"q4_k": M.TYPE_Q4_K, "q6_k": M.TYPE_Q6_K, "q8_0": M.TYPE_Q8_0, "q5_0": M.TYPE_Q5_0,
         "q4_0": M.TYPE_Q4_0, "f16": M.TYPE_F16}
BLOCK = {"q4_k": (256, 144), "q6_k": (256, 210), "q8_0": (32, 34), "q5_0": (32, 22), "q4_0": (32, 18),
         "f16": (32, 64)}
ACTS = {"silu": M.ACT_SILU, "gelu_erf_gp1": M.ACT_GELU_ERF_GP1, "gelu_tanh": M.ACT_GELU_TANH,
        "relu_sqr": M.ACT_RELU_SQR}
MODELS = {
    "moondream3": dict(D=2048, E=64, K=8, I=1024, fused=True, gated=True, act="gelu_erf_gp1", norm=M.NORM_LAYER,
                       gating=M.GATING_SOFTMAX_TOPK, shared=0),
    "qwen3omni": dict(D=2048, E=128, K=8, I=768, fused=False, gated=True, act="silu", norm=M.NORM_RMS,
                      gating=M.GATING_SOFTMAX_TOPK, shared=0),
    "diffusiongemma": dict(D=2816, E=128, K=8, I=704, fused=False, gated=True, act="gelu_tanh", norm=M.NORM_RMS,
                           gating=M.GATING_SOFTMAX_ALL, shared=0),
    "nemotronomni": dict(D=2688, E=128, K=6, I=1856, fused=False, gated=False, act="relu_sqr", norm=M.NORM_RMS,
                         gating=M.GATING_SIGMOID_BIAS, shared=3712),
}
EPS = 1e-6
SCALING = 2.5       # nemotronomni's factor on the renormalized weights
GATE_EPS = 1e-20
ZIPF_IDLE = 16


def _case(name, model, op, T, gate, down=None, layers=1, act=None, tiled=False, zipf=False, routing=False):
    return {"name": name, "model": model, "op": op, "T": T, "layers": layers, "gate": gate, "down": down or gate,
            "act": act or MODELS[model]["act"], "tiled": tiled, "zipf": zipf, "routing": routing}


def listed():
    return [
        # one token through the MoE blocks of a 24-layer stack: the inner loop of text generation
        _case("decode_1_stack24", "moondream3", "norm", 1, "q4_k", layers=24),
        # one token whose experts the host's expert cache chose (ids and weights from the caller)
        _case("decode_1_caller_ids", "qwen3omni", "caller_ids", 1, "q4_k", layers=8),
        # eight sequences decoded together
        _case("decode_8", "qwen3omni", "norm", 8, "q4_k", tiled=True),
        # a larger ragged decode batch on the tables as the file holds them
        _case("decode_33_rows", "qwen3omni", "norm", 33, "q4_k"),
        # a short prompt, an image's tokens or a prefill chunk
        _case("prefill_301", "qwen3omni", "norm", 301, "q4_k", tiled=True),
        # the library's headline workload: a 1024-token prefill
        _case("prefill_1024", "moondream3", "forward", 1024, "q4_k", "q6_k", act="gelu_tanh", tiled=True),
        # a long prefill with hot and idle experts, on the file's tables, the caller reading the routing
        _case("prefill_2000_skewed", "moondream3", "forward", 2000, "q4_k", "q6_k", zipf=True, routing=True),
        # the higher-quality k-quant file
        _case("prefill_509_q6_k", "moondream3", "norm", 509, "q6_k"),
        # the converters' default file type: a small decode batch and a prefill
        _case("decode_5_q8_0", "qwen3omni", "norm", 5, "q8_0"),
        _case("prefill_600_q8_0", "moondream3", "norm", 600, "q8_0"),
        # a block of 256 positions denoised together, unquantized tables, router on its own rows
        _case("canvas_256_f16", "diffusiongemma", "own_router", 256, "f16"),
        # a batch through relu^2 experts, the sigmoid router and the shared expert
        _case("batch_200_q5_0_shared", "nemotronomni", "norm", 200, "q5_0"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    kind = rng.choice(["stack", "caller", "decode", "prefill", "prefill", "q6_k", "b32", "b32", "canvas", "shared"])
    model = rng.choice(["moondream3", "qwen3omni"])
    down = rng.choice(["q4_k", "q6_k"]) if model == "moondream3" else "q4_k"
    tiled = rng.random() < 0.5
    if kind == "stack":
        c = _case("", model, "norm", 1, "q4_k", down, layers=rng.randint(6, 24))
    elif kind == "caller":
        t = rng.choice(["q4_k", "q4_k", "q8_0"])
        c = _case("", model, "caller_ids", _log_int(rng, 1, 4), t, layers=rng.randint(4, 12))
    elif kind == "decode":
        c = _case("", model, "norm", _log_int(rng, 2, 64), "q4_k", down, tiled=tiled)
    elif kind == "prefill":
        c = _case("", model, rng.choice(["norm", "forward"]), _log_int(rng, 65, 1800), "q4_k", down, tiled=tiled,
                  act=rng.choice(["gelu_erf_gp1", "gelu_tanh"]) if model == "moondream3" else None,
                  zipf=model == "moondream3" and rng.random() < 0.3, routing=rng.random() < 0.3)
    elif kind == "q6_k":
        c = _case("", model, "norm", _log_int(rng, 1, 700), "q6_k")
    elif kind == "b32":
        c = _case("", model, "norm", _log_int(rng, 1, 600), rng.choice(["q8_0", "q8_0", "q5_0", "q4_0", "f16"]))
    elif kind == "canvas":
        c = _case("", "diffusiongemma", "own_router", _log_int(rng, 1, 256), rng.choice(["f16", "q4_0", "q8_0"]))
    else:
        c = _case("", "nemotronomni", "norm", _log_int(rng, 1, 200), rng.choice(["q5_0", "q8_0"]))
    del c["name"]
    return c


# ---------------------------------------------------------------- tables
def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _quantize(kind, w):
    """w [..., K] float32 -> (rows [..., row bytes] uint8, the rows' values in float64 as a function)."""
    lead, (n, size) = w.shape[:-1], BLOCK[kind]
    b = w.reshape(*lead, -1, n)
    if kind == "f16":
        h = b.half()
        return _bytes(h).reshape(*lead, -1), lambda: h.to(F64).reshape(w.shape)
    if kind == "q8_0":
        d = (b.abs().amax(-1, keepdim=True) / 127.0).half()
        q = torch.round(b / d.float().clamp_min(1e-8)).clamp_(-127, 127).to(torch.int8)
        raw = torch.cat([_bytes(d), _bytes(q)], -1)
        return raw.reshape(*lead, -1), lambda: (d.to(F64) * q.to(F64)).reshape(w.shape)
    if kind in ("q5_0", "q4_0"):
        half = 16 if kind == "q5_0" else 8
        d = (b.abs().amax(-1, keepdim=True) / (half - 0.5)).half()
        q = (torch.round(b / d.float().clamp_min(1e-8)) + half).clamp_(0, 2 * half - 1).to(torch.int32)
        nib = ((q[..., :16] & 15) | ((q[..., 16:] & 15) << 4)).to(torch.uint8)
        parts = [_bytes(d), nib]
        if kind == "q5_0":
            bits = ((q >> 4).to(torch.int64) << torch.arange(32, device=q.device)).sum(-1, keepdim=True)
            parts.insert(1, ((bits >> torch.tensor([0, 8, 16, 24], device=q.device)) & 255).to(torch.uint8))
        return torch.cat(parts, -1).reshape(*lead, -1), lambda: (d.to(F64) * (q - half).to(F64)).reshape(w.shape)
    if kind == "q4_k":
        s = b.unflatten(-1, (8, 32))
        lo = s.amin(-1).clamp_max(0.0)
        span = (s.amax(-1) - lo) / 15.0
        d = (span.amax(-1, keepdim=True) / 63.0).half()
        dm = ((-lo).amax(-1, keepdim=True) / 63.0).half()
        sc = torch.round(span / d.float().clamp_min(1e-8)).clamp_(0, 63)
        mn = torch.round(-lo / dm.float().clamp_min(1e-8)).clamp_(0, 63)
        step = (d.float() * sc)[..., None]
        q = torch.round((s + (dm.float() * mn)[..., None]) / step.clamp_min(1e-12)).clamp_(0, 15).to(torch.uint8)
        si, mi = sc.to(torch.int32), mn.to(torch.int32)
        packed = torch.cat([(si[..., :4] & 63) | ((si[..., 4:] >> 4) << 6), (mi[..., :4] & 63) | ((mi[..., 4:] >> 4) << 6),
                            (si[..., 4:] & 15) | ((mi[..., 4:] & 15) << 4)], -1).to(torch.uint8)
        nib = (q[..., 0::2, :] | (q[..., 1::2, :] << 4)).flatten(-2)
        raw = torch.cat([_bytes(d), _bytes(dm), packed, nib], -1)
        return raw.reshape(*lead, -1), lambda: ((d.to(F64) * sc.to(F64))[..., None] * q.to(F64)
                                                - (dm.to(F64) * mn.to(F64))[..., None]).reshape(w.shape)
    s = b.unflatten(-1, (16, 16))                     # q6_k
    step = s.abs().amax(-1) / 31.0
    d = (step.amax(-1, keepdim=True) / 127.0).half()
    sc = torch.round(step / d.float().clamp_min(1e-8)).clamp_(0, 127)
    full = (d.float() * sc)[..., None]
    q = torch.round(s / full.clamp_min(1e-12)).clamp_(-32, 31)
    u = (q.to(torch.int32) + 32).flatten(-2).unflatten(-1, (2, 4, 32))   # halves of four 32-value quarters
    ql = torch.cat([(u[..., 0, :] & 15) | ((u[..., 2, :] & 15) << 4), (u[..., 1, :] & 15) | ((u[..., 3, :] & 15) << 4)],
                   -1).flatten(-2).to(torch.uint8)
    qh = ((u[..., 0, :] >> 4) | ((u[..., 1, :] >> 4) << 2) | ((u[..., 2, :] >> 4) << 4)
          | ((u[..., 3, :] >> 4) << 6)).flatten(-2).to(torch.uint8)
    raw = torch.cat([ql, qh, _bytes(sc.to(torch.int8)), _bytes(d)], -1)
    return raw.reshape(*lead, -1), lambda: ((d.to(F64) * sc.to(F64))[..., None] * q.to(F64)).reshape(w.shape)


def _gen(seed, *salt):
    v = seed
    for s in salt:
        v = (v * 1000003 + s + 1) % (1 << 62)
    return torch.Generator(device="cuda").manual_seed(v)


def _normal(shape, seed, *salt, std=1.0):
    return torch.randn(shape, generator=_gen(seed, *salt), device="cuda") * std


def _table(kind, E, N, K, seed, salt, values=False, only=None):
    """An expert table [E][N rows of K]: its bytes, or its values (a dict of the experts in `only`)."""
    step, got = max(1, (1 << 26) // (N * K)), []
    vals = {}
    for e in range(0, E, step):
        n = min(step, E - e)
        raw, value = _quantize(kind, _normal((n, N, K), seed, salt, e, std=0.02))
        if not values:
            got.append(raw)
            continue
        if only is None or any(e <= i < e + n for i in only):
            v = value()
            for i in range(n):
                if only is None or e + i in only:
                    vals[e + i] = v[i].clone()
    return vals if values else torch.cat(got)


def _inputs(case, seed, layer):
    """The layer's small tensors and the step's rows."""
    m, T = MODELS[case["model"]], case["T"]
    D, E, K = m["D"], m["E"], m["K"]
    # rows of a residual stream: channels of different sizes, a few of them large
    size = torch.exp(0.4 * _normal((D,), seed, layer, 1))
    size[torch.randperm(D, generator=_gen(seed, layer, 2), device="cuda")[:4]] *= 8.0
    h = _normal((T, D), seed, layer, 3) * size
    t = {"h": h, "router_w": _normal((E, D), seed, layer, 4, std=0.02)}
    # normalized rows, for the entry points that take them as input
    t["x"] = (h / torch.sqrt((h * h).mean(-1, keepdim=True) + EPS)) * (1.0 + 0.1 * _normal((D,), seed, layer, 5))
    if case["op"] == "norm":
        t["norm_w"] = 1.0 + 0.1 * _normal((D,), seed, layer, 5)
        if m["norm"] == M.NORM_LAYER:
            t["norm_b"] = 0.05 * _normal((D,), seed, layer, 6)
    if case["op"] == "own_router":
        t["x_router"] = _normal((T, D), seed, layer, 7)
    if case["op"] == "caller_ids":
        t["ids"] = torch.rand((T, E), generator=_gen(seed, layer, 8), device="cuda").argsort(-1)[:, :K].int().contiguous()
        t["w"] = torch.softmax(_normal((T, K), seed, layer, 9), -1)
    if case["zipf"]:
        live = E - ZIPF_IDLE
        p = torch.arange(1, live + 1, device="cuda", dtype=F64) ** -1.2
        bias = torch.full((E,), -1.0e4, device="cuda")
        bias[torch.randperm(E, generator=_gen(seed, layer, 10), device="cuda")[:live]] = (0.8 * torch.log(p / p.sum())).float()
        t["router_b"] = bias
    if m["gating"] == M.GATING_SIGMOID_BIAS:
        t["sel_bias"] = _normal((E,), seed, layer, 11, std=0.05)
    if m["gating"] == M.GATING_SOFTMAX_ALL:
        t["expert_scale"] = 0.5 + torch.rand((E,), generator=_gen(seed, layer, 12), device="cuda")
    return t


def _tables(case, seed, layer, **kw):
    """name -> table of the layer's expert tables (bytes, or values with values=True)."""
    m = MODELS[case["model"]]
    D, E, I, s = m["D"], m["E"], m["I"], seed * 64 + layer
    up = 2 * I if m["fused"] else I
    t = {"gate": _table(case["gate"], E, up, D, s, 1, **kw), "down": _table(case["down"], E, D, I, s, 2, **kw)}
    if m["gated"] and not m["fused"]:
        t["up"] = _table(case["gate"], E, I, D, s, 3, **kw)
    if m["shared"]:
        kw.pop("only", None)
        t["sh_gate"] = _table(case["gate"], 1, m["shared"], D, s, 4, **kw)
        t["sh_down"] = _table(case["down"], 1, D, m["shared"], s, 5, **kw)
    return t


# ---------------------------------------------------------------- the calls
def prepare(case, seed):
    m, T = MODELS[case["model"]], case["T"]
    D, E, K, I = m["D"], m["E"], m["K"], m["I"]
    ctx = M.Context(0)
    ctx.reserve(T, D, I, E, K)
    state = {"op": case["op"], "ctx": ctx, "T": T, "layers": []}
    for n in range(case["layers"]):
        t, q = _inputs(case, seed, n), _tables(case, seed, n)
        if case["op"] == "own_router":
            t["res"] = t.pop("h")

        def tensor(name, kind, ne):
            return M.tensor(q[name].data_ptr(), TYPES[kind], ne)

        up_rows = 2 * I if m["fused"] else I
        layer = M.make_layer(D, E, K, I, t["router_w"].data_ptr(), t["router_b"].data_ptr() if "router_b" in t else None,
                             tensor("gate", case["gate"], [D, up_rows, E]),
                             tensor("up", case["gate"], [D, I, E]) if "up" in q else None,
                             tensor("down", case["down"], [I, D, E]), m["fused"], ACTS[case["act"]])
        layer.gating = m["gating"]
        if m["gating"] == M.GATING_SIGMOID_BIAS:
            layer.sel_bias, layer.routed_scaling, layer.gate_eps = t["sel_bias"].data_ptr(), SCALING, GATE_EPS
        if m["gating"] == M.GATING_SOFTMAX_ALL:
            layer.expert_scale = t["expert_scale"].data_ptr()
        if m["shared"]:
            layer.sh_n_ff, layer.sh_act = m["shared"], M.ACT_RELU_SQR
            layer.sh_gate = tensor("sh_gate", case["gate"], [D, m["shared"]])
            layer.sh_down = tensor("sh_down", case["down"], [m["shared"], D])
        if case["tiled"]:
            for name in [k for k in ("gate", "up", "down") if k in q]:
                src = getattr(layer, name)
                q[name + "_tiled"] = torch.empty(M.tiled_bytes(src), dtype=torch.uint8, device="cuda")
                desc = M.Tensor()
                M.check("mi_moe_tile", ctx.tile(src, q[name + "_tiled"].data_ptr(), desc))
                setattr(layer, name + "_tiled", desc)
        norm = None
        if case["op"] == "norm":
            norm = M.make_norm(m["norm"], EPS, t["norm_w"].data_ptr(), t["norm_b"].data_ptr() if "norm_b" in t else None)
        t["out"] = torch.empty((T, D), device="cuda")
        routing = None
        if case["routing"]:
            routing = M.Routing()
            t["sel"] = torch.empty((T, K), dtype=torch.int32, device="cuda")
            t["weights"] = torch.empty((T, K), device="cuda")
            t["counts"] = torch.empty((E,), dtype=torch.int32, device="cuda")
            for k in ("sel", "weights", "counts"):
                setattr(routing, k, ctypes.c_void_p(t[k].data_ptr()))
        state["layers"].append({"layer": layer, "norm": norm, "routing": routing, "t": t, "tables": q})
    torch.cuda.synchronize()
    return state


def run(state):
    ctx, T, op = state["ctx"], state["T"], state["op"]
    stream = torch.cuda.current_stream().cuda_stream
    outs = []
    for s in state["layers"]:
        t, layer = s["t"], s["layer"]
        out = t["out"].data_ptr()
        if op == "norm":
            h = t["h"].data_ptr()
            rc = ctx.forward_norm(layer, s["norm"], h, T, h, out, s["routing"], stream)
        elif op == "forward":
            rc = ctx.forward(layer, t["x"].data_ptr(), T, t["h"].data_ptr(), out, s["routing"], stream)
        elif op == "own_router":
            rc = ctx.forward_router_input(layer, t["x"].data_ptr(), t["x_router"].data_ptr(), T, t["res"].data_ptr(), out,
                                          s["routing"], stream)
        else:
            ids = t["ids"].data_ptr()
            rc = ctx.expert_ffn(layer, t["x"].data_ptr(), T, None, ids, ids, t["w"].data_ptr(), out, stream)
        M.check(op, rc)
        outs.append(t["out"])
        if s["routing"] is not None:
            outs += [t["sel"], t["weights"], t["counts"]]
    return outs


def _row_bytes(kind, n):
    return n // BLOCK[kind][0] * BLOCK[kind][1]


def work(case):
    m, T, L = MODELS[case["model"]], case["T"], case["layers"]
    D, E, K, I = m["D"], m["E"], m["K"], m["I"]
    live = E - ZIPF_IDLE if case["zipf"] else E
    hit = live * (1.0 - (1.0 - K / live) ** T)       # experts that a token chose, evenly spread
    products = 2 if m["gated"] else 1
    per_expert = products * I * _row_bytes(case["gate"], D) + D * _row_bytes(case["down"], I)
    rows = 3 + (case["op"] == "own_router") - (case["op"] == "caller_ids")   # x or h, res, out
    if case["op"] == "norm":
        rows = 2
    b = hit * per_expert + 4.0 * rows * T * D
    f = 2.0 * T * K * (products + 1) * D * I
    if case["op"] != "caller_ids":
        b += 4.0 * E * D
        f += 2.0 * T * E * D
    if m["shared"]:
        b += m["shared"] * _row_bytes(case["gate"], D) + D * _row_bytes(case["down"], m["shared"])
        f += 4.0 * T * D * m["shared"]
    return {"bytes": L * b, "flops": L * f}


def tolerance(case):
    """The products start with an 8-bit rounding of the activations (ggml's Q8_K / Q8_0), once of x and once of the
    rows between the two products, where a value that differs in its last bits moves a code by one step; the matrix
    units' operands are 16-bit.  Measured against float64: 0.001 - 0.009 of a result that holds the residual stream,
    0.02 - 0.03 without it (two products that agree on the codes but for single steps are four times nearer to each
    other).  F16 tables: the rows' rounding to fp16 alone, measured 5e-5."""
    if case["gate"] == "f16":
        return {"rel": 2e-4, "max": 4e-3, "differ": 1e-3}
    if case["op"] == "caller_ids":
        return {"rel": 3e-2, "max": 3e-1, "differ": 1e-3}
    return {"rel": 1e-2, "max": 1e-1, "differ": 1e-3}


# ---------------------------------------------------------------- in float64, from the definitions
def _activate(act, a, b):
    if act == "relu_sqr":
        return torch.relu(a) ** 2
    if act == "silu":
        return a * torch.sigmoid(a) * b
    if act == "gelu_tanh":
        return 0.5 * a * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (a + 0.044715 * a ** 3))) * b
    return 0.5 * a * (1.0 + torch.erf(a / math.sqrt(2.0))) * (b + 1.0)


def _norm64(kind, h, w, b):
    if kind == M.NORM_RMS:
        return h / torch.sqrt((h * h).mean(-1, keepdim=True) + EPS) * w
    d = h - h.mean(-1, keepdim=True)
    y = d / torch.sqrt((d * d).mean(-1, keepdim=True) + EPS) * w
    return y if b is None else y + b


def _route64(m, t, xr):
    logits = xr @ t["router_w"].T + (t["router_b"] if "router_b" in t else 0.0)
    p = logits
    if m["gating"] == M.GATING_SIGMOID_BIAS:
        p = torch.sigmoid(logits)
        ids = torch.sort(p + t["sel_bias"], dim=-1, descending=True, stable=True)[1][:, :m["K"]]
        w = p.gather(1, ids)
        return ids, w / (w.sum(-1, keepdim=True) + GATE_EPS) * SCALING
    ids = torch.sort(logits, dim=-1, descending=True, stable=True)[1][:, :m["K"]]
    w = torch.softmax(logits.gather(1, ids), -1)
    return ids, w * t["expert_scale"][ids] if "expert_scale" in t else w


def exact(case, seed):
    m, outs = MODELS[case["model"]], []
    I = m["I"]
    for n in range(case["layers"]):
        t = {k: v if k == "ids" else v.to(F64) for k, v in _inputs(case, seed, n).items()}
        x, res = t["x"], t["h"]
        if case["op"] == "norm":
            x = _norm64(m["norm"], t["h"], t["norm_w"], t.get("norm_b"))
        if case["op"] == "caller_ids":
            ids, w, res = t["ids"].long(), t["w"], 0.0
        else:
            ids, w = _route64(m, t, t.get("x_router", x))
        used = sorted(set(ids.flatten().tolist()))
        v = _tables(case, seed, n, values=True, only=set(used))
        out = torch.zeros_like(x)
        for e in used:
            rows, slot = torch.nonzero(ids == e, as_tuple=True)
            a = x[rows] @ v["gate"][e].T
            if m["fused"]:
                a = _activate(case["act"], a[:, :I], a[:, I:])
            else:
                a = _activate(case["act"], a, x[rows] @ v["up"][e].T if "up" in v else None)
            out.index_add_(0, rows, (a @ v["down"][e].T) * w[rows, slot][:, None])
        if m["shared"]:
            out += _activate("relu_sqr", x @ v["sh_gate"][0].T, None) @ v["sh_down"][0].T
        outs.append(out + res)
        if case["routing"]:
            outs += [ids.int(), w, torch.bincount(ids.flatten(), minlength=m["E"]).int()]
    return outs
