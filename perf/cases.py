"""The work that is timed: what a program that trains or serves a routed-experts layer
has the library do, through its public entry points (bux_amd.moe, bux_amd.router,
bux_amd.dispatch), over the sizes that its configurations, tests and benchmark use.

A case is a dict of plain values. Its `kind`:

- "layer": the routed experts, `moe.experts_forward`, and with `step` the backward too
  (`moe.experts_backward`); `fmt` mxfp8, mxfp8_2d or compute, bfloat16 or float32 tokens;
  `given` the kernels already in MXFP8; `fprop` the forward pass alone in MXFP8 (a
  serving program: no gradients follow); `graph` the call captured once in a HIP graph
  and replayed, as a program does whose calls are shorter than their launches; `skew`
  how the picks fall on the experts.
- "route": the router's top-k, `router.route`.
- "dispatch": an expert-parallel exchange's rows, packed by pick and unpacked.
- "weights": the experts' kernels to MXFP8 (`moe.in_mxfp8`), once an optimizer step.
"""

import math

import torch

BF16 = torch.bfloat16

_LAYER = {"kind": "layer", "step": False, "graph": False, "fmt": "mxfp8", "dtype": "bfloat16",
          "skew": "even", "activation": "swish", "limit": 0.0, "offset": 0.0, "bias": False,
          "norm": False, "given": False, "fprop": False}


def _layer(**kw):
    return {**_LAYER, **kw}


QWEN3 = {"d": 2048, "experts": 128, "k": 8, "f": 768}  # Qwen3-30B-A3B's experts
GPT_OSS = {"d": 2880, "experts": 128, "k": 4, "f": 2880}  # gpt-oss-120b's
DEEPSEEK = {"d": 7168, "experts": 256, "k": 8, "f": 2048}  # DeepSeek-V3's


def listed():
    return [
        # a decode step of a small batch: few rows, most of them alone with their expert
        _layer(name="decode 8", tokens=8, graph=True, given=True, fprop=True, **QWEN3),
        # a larger decode batch, or a short prompt: every expert's weights, a dozen rows each
        _layer(name="decode 200", tokens=200, graph=True, given=True, fprop=True, **QWEN3),
        # the tiny bfloat16 layer, called eagerly: launches and host work
        _layer(name="tiny bf16 forward", tokens=4096, d=256, experts=8, k=2, f=512, fmt="compute"),
        # the router of a whole batch of tokens
        {"name": "route", "kind": "route", "tokens": 16384, "d": 2048, "experts": 128, "k": 8,
         "router": "softmax", "groups": 1, "top_groups": 1, "scaling": 1.0},
        # an expert-parallel exchange: the picks' rows out, and back to bfloat16
        {"name": "dispatch", "kind": "dispatch", "tokens": 16384, "d": 2048, "experts": 128, "k": 8},
        # every expert's kernels to MXFP8 after an optimizer step
        {"name": "weights to mxfp8", "kind": "weights", "fmt": "mxfp8", "d": 2048, "experts": 128,
         "f": 768},
        # a gpt-oss-120b layer's forward: biases, clamped gated activation, uneven experts
        _layer(name="gpt-oss forward", tokens=8192, given=True, skew="biased", bias=True,
               activation="quick_gelu", limit=7.0, offset=1.0, **GPT_OSS),
        # a DeepSeek-V3 layer's forward on Zipf loads: experts of 0 to 8192 rows
        _layer(name="deepseek forward", tokens=8192, given=True, skew="zipf", **DEEPSEEK),
        # the headline: a Qwen3-30B-A3B layer's training step
        _layer(name="qwen3 step", tokens=16384, step=True, **QWEN3),
        # a micro-batch of it between two optimizer steps: the kernels are in MXFP8 already
        _layer(name="qwen3 micro-batch step", tokens=2000, step=True, given=True, **QWEN3),
        # the same layer trained in bfloat16
        _layer(name="qwen3 bf16 step", tokens=8192, step=True, fmt="compute", **QWEN3),
        # a float32 layer with biases and a norm of the experts' outputs, an odd batch
        _layer(name="float32 step", tokens=1001, step=True, dtype="float32", d=1024, experts=16,
               k=4, f=512, bias=True, norm=True),
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread evenly over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["layer", "route", "dispatch", "weights"], [9, 1, 1, 1])[0]
    d = 32 * _log_int(rng, 4, 224)
    experts = rng.choice([8, 16, 32, 60, 64, 96, 128, 160, 256])
    k = rng.choice([1, 2, 4, 6, 8])
    if kind == "route":
        grouped = experts % 8 == 0 and experts >= 64 and rng.random() < 0.3
        return {"kind": kind, "tokens": _log_int(rng, 1, 32768), "d": 64 * _log_int(rng, 2, 112),
                "experts": experts, "k": k, "router": "sigmoid" if grouped else "softmax",
                "groups": 8 if grouped else 1, "top_groups": 4 if grouped else 1,
                "scaling": 2.5 if grouped else 1.0}
    if kind == "dispatch":
        most = max(1, min(16384, (1 << 28) // (d * k)))
        return {"kind": kind, "tokens": _log_int(rng, 1, most), "d": d, "experts": experts, "k": k}
    f = 32 * _log_int(rng, 4, 128)
    while experts * d * f > 4e8:  # at most twice the weights of the largest training step
        experts = max(8, experts // 2)
        if experts == 8:
            f = max(128, f // 64 * 32)
    if kind == "weights":
        return {"kind": kind, "fmt": rng.choice(["mxfp8", "mxfp8", "mxfp8_2d"]), "d": d,
                "experts": experts, "f": f}
    dtype = "float32" if rng.random() < 0.15 else "bfloat16"
    fmt = rng.choices(["mxfp8", "mxfp8_2d", "compute"], [7, 1, 2])[0]
    step = rng.random() < 0.5
    serve = not step and fmt == "mxfp8" and rng.random() < 0.5
    most = 3e12 if fmt != "compute" else 1.2e12
    if dtype == "float32" and fmt == "compute":
        most = 5e10
    most = int(min(16384, 131072 // k, most / (6 * k * d * f * (3 if step else 1))))
    act, limit, offset = rng.choice([("swish", 0.0, 0.0), ("swish", 0.0, 0.0),
                                     ("quick_gelu", 7.0, 1.0)])
    return _layer(tokens=_log_int(rng, 1, max(1, most)), d=d, experts=experts, k=k, f=f, step=step,
                  graph=serve, given=serve or (fmt != "compute" and rng.random() < 0.5),
                  fprop=serve, fmt=fmt, dtype=dtype, skew=rng.choice(["even", "biased", "zipf"]),
                  activation=act, limit=limit, offset=offset, bias=rng.random() < 0.2,
                  norm=rng.random() < 0.1)


# --- inputs ------------------------------------------------------------------------------


def _dtype(case):
    return torch.float32 if case.get("dtype") == "float32" else BF16


def _normal(gen, shape, scale, dtype):
    """Normal values of `dtype`, made a slice at a time (the experts' kernels are large)."""
    out = torch.empty(shape, dtype=dtype, device="cuda")
    if len(shape) < 3:
        return out.copy_(torch.randn(shape, generator=gen, device="cuda") * scale)
    for part in out:
        part.copy_(torch.randn(part.shape, generator=gen, device="cuda") * scale)
    return out


def _tokens(gen, case):
    """N(0, 1) with a thousandth of the values 100 times as large."""
    t, d = case["tokens"], case["d"]
    z = torch.randn(t, d, generator=gen, device="cuda")
    at = torch.randint(t * d, (max(1, t * d // 1000),), generator=gen, device="cuda")
    z.view(-1)[at] *= 100
    return z.to(_dtype(case))


def _picks(gen, case):
    """Each token's k experts and their softmax weights, normalised: router logits N(0, 1),
    "biased" with each expert's own offset N(0, 0.5); "zipf": the experts' shares as
    1 / rank^1.2, the last fifth of the ranks empty (picks drawn without replacement)."""
    t, e, k = case["tokens"], case["experts"], case["k"]
    skew = case.get("skew", "even")
    logits = torch.randn(t, e, generator=gen, device="cuda")
    if skew == "biased":
        logits += 0.5 * torch.randn(e, generator=gen, device="cuda")
    if skew == "zipf":
        rank = torch.randperm(e, generator=gen, device="cuda").float()
        live = max(k, e - round(e * 0.2))
        share = torch.where(rank < live, -1.2 * torch.log1p(rank), -torch.inf)
        u = torch.rand(t, e, generator=gen, device="cuda").clamp_(1e-7, 1 - 1e-7)
        idx = torch.topk(share - torch.log(-torch.log(u)), k, -1).indices
        w = torch.softmax(torch.gather(logits, 1, idx), -1)
    else:
        w, idx = torch.topk(torch.softmax(logits, -1), k, -1)
        w = w / w.sum(-1, keepdim=True)
    return idx.to(torch.int32).contiguous(), w.to(_dtype(case))


def _kernels(gen, case):
    e, d, f = case["experts"], case["d"], case["f"]
    dt = _dtype(case)
    return _normal(gen, (e, d, f, 2), 0.02, dt), _normal(gen, (e, f, d), 0.02, dt)


def _inputs(case, seed):
    """A layer's inputs, by name."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = _dtype(case)
    e, d, f = case["experts"], case["d"], case["f"]
    z = _tokens(gen, case)
    idx, w = _picks(gen, case)
    up, down = _kernels(gen, case)
    given = {"z": z, "idx": idx, "weights": w, "up": up, "down": down}
    given["dy"] = _normal(gen, (case["tokens"], d), 1e-2, dt) if case["step"] else None
    given["up_bias"] = _normal(gen, (e, f * 2), 0.1, dt).view(e, f, 2) if case["bias"] else None
    given["down_bias"] = _normal(gen, (e, d), 0.1, dt) if case["bias"] else None
    given["norm_scale"] = (1 + _normal(gen, (1, d), 0.1, dt)).view(d) if case["norm"] else None
    return given


def _forward(case, x, quantized):
    from bux_amd import moe
    ffn = moe.Ffn(case["activation"], case["limit"] or None, case["offset"])
    norm = moe.ExpertNorm("rmsnorm") if case["norm"] else None
    out, saved = moe.experts_forward(
        x["z"], x["idx"], x["weights"], x["up"], x["down"], ffn, case["fmt"], quantized=quantized,
        passes=("fprop",) if case["fprop"] else None, up_bias=x["up_bias"],
        down_bias=x["down_bias"], norm=norm, norm_scale=x["norm_scale"])
    if not case["step"]:
        return {"out": out}
    grads = moe.experts_backward(saved, x["dy"], x["up"], x["down"], ffn, case["fmt"],
                                 up_bias=x["up_bias"], down_bias=x["down_bias"], norm=norm,
                                 norm_scale=x["norm_scale"])
    return {"out": out, **{name: g for name, g in grads.items() if g is not None}}


def prepare(case, seed):
    from bux_amd import moe
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case}
    if case["kind"] == "route":
        state["z"] = _tokens(gen, case)
        state["kernel"] = _normal(gen, (case["d"], case["experts"]), 0.02, BF16)
        state["router_bias"] = (0.1 * torch.randn(case["experts"], generator=gen, device="cuda")
                                if case["groups"] > 1 else None)
    elif case["kind"] == "dispatch":
        state["z"] = _tokens(gen, case)
        state["order"] = moe.sort_by_expert(_picks(gen, case)[0], case["experts"]).order
    elif case["kind"] == "weights":
        state["up"], state["down"] = _kernels(gen, case)
    else:
        state["x"] = x = _inputs(case, seed)
        state["quantized"] = moe.in_mxfp8(x["up"], x["down"], case["fmt"]) if case["given"] else None
        if case["graph"]:
            _capture(state)
    return state


def _capture(state):
    """The layer's call in a HIP graph over the state's inputs: a warm-up on a stream of
    its own, then the capture."""
    case, x, quantized = state["case"], state["x"], state["quantized"]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _forward(case, x, quantized)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    state["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(state["graph"]):
        state["outputs"] = _forward(case, x, quantized)


def run(state):
    from bux_amd import dispatch, moe, router
    case = state["case"]
    if case["kind"] == "route":
        r = router.route(state["z"], state["kernel"], top_k=case["k"], router=case["router"],
                         router_bias=state["router_bias"], num_groups=case["groups"],
                         top_k_groups=case["top_groups"], routed_scaling_factor=case["scaling"])
        return {"idx": r.idx, "weights": r.weights}
    if case["kind"] == "dispatch":
        packed = dispatch.picked_in_mxfp8(state["z"], state["order"], case["k"])
        return {"packed": packed, "rows": dispatch.from_mxfp8(packed, case["d"])}
    if case["kind"] == "weights":
        q = moe.in_mxfp8(state["up"], state["down"], case["fmt"])
        return {name: list(getattr(q, name)) for name in ("up_n", "up_k", "down_n", "down_k")}
    if case["graph"]:
        state["graph"].replay()
        return state["outputs"]
    return _forward(case, state["x"], state["quantized"])


# --- what a pass cannot do without -------------------------------------------------------


def work(case):
    d, e = case["d"], case["experts"]
    q = 1 + 1 / 32  # an E4M3 code and its share of a scale byte
    if case["kind"] == "weights":
        return {"bytes": 3 * e * d * case["f"] * (2 + 2 * q), "flops": 0}
    t, k = case["tokens"], case["k"]
    m = t * k
    if case["kind"] == "route":
        return {"bytes": 2 * t * d + 2 * d * e + 6 * m, "flops": 2 * t * d * e}
    if case["kind"] == "dispatch":
        return {"bytes": 2 * t * d + 4 * m + m * d * (q + 2), "flops": 0}
    f, s = case["f"], 4 if case["dtype"] == "float32" else 2
    live = e - round(e * 0.2) if case["skew"] == "zipf" else e
    touched = live * (1 - (1 - 1 / live) ** m)  # experts with a row, about
    kernels = touched * 3 * d * f * (q if case["given"] else s)
    total = 2 * t * d * s + m * (4 + s) + kernels
    if case["step"]:  # dy and the kernels along their other axis in, the gradients out
        total += 2 * t * d * s + m * s + 3 * e * d * f * s + (kernels if case["given"] else 0)
    return {"bytes": total, "flops": 6 * m * d * f * (3 if case["step"] else 1)}


def tolerance(case):
    if case["kind"] in ("weights", "dispatch"):
        return "exact"
    if case["kind"] == "route":  # bfloat16 weights; picks whose scores tie within a float32 sum
        return {"rel": 1e-3, "max": 0.05, "differ": 2e-3}
    if case["fmt"] == "compute":
        return {"rel": 2e-5, "max": 1e-3} if case["dtype"] == "float32" else {"rel": 2e-3, "max": 0.3}
    # a last bit of a float32 sum flips a bfloat16 rounding and then an E4M3 code after it
    return {"rel": 2e-2 if case["norm"] else 1e-2, "max": 0.8}


# --- the same in 64 bits -----------------------------------------------------------------


def _rounded(x, dt):
    """x (float64) as the layer stores it: rounded once to its dtype."""
    return x.to(dt).double()


def _blocks(x, square=False):
    """x's values in MXFP8 along its rows, blocks of 32 (`square`: 32 x 32 tiles)."""
    r, c = x.shape
    cp, rp = -(-c // 32) * 32, -(-r // 32) * 32 if square else r
    v = torch.nn.functional.pad(x, (0, cp - c, 0, rp - r))
    v = v.view(rp // 32, 32, cp // 32, 32) if square else v.view(r, cp // 32, 32)
    top = v.abs().amax(dim=(1, 3) if square else 2, keepdim=True).float() / 448.0
    mantissa, exponent = torch.frexp(top)
    exponent = exponent - (mantissa == 0.5).to(exponent.dtype)
    exponent = torch.where(top == 0, -126, exponent).clamp(-126, 126).double()
    scale = torch.exp2(exponent)
    codes = (v / scale).clamp(-448, 448).float().to(torch.float8_e4m3fn).double()
    return (codes * scale).reshape(rp, cp)[:r, :c]


def _activation(case, projected, w):
    """h (m, f) of projected (m, 2 f), (up, gate) pairs, and the rows' weights, unrounded."""
    pair = projected.view(projected.shape[0], -1, 2)
    up, gate = pair[..., 0], pair[..., 1]
    if case["limit"]:  # minimum and maximum halve the gradient at a tie, as the layer does
        limit = torch.full_like(up, case["limit"])
        up, gate = torch.minimum(torch.maximum(up, -limit), limit), torch.minimum(gate, limit)
    alpha = 1.0
    if case["activation"] == "quick_gelu":  # 1.702 in the layer's dtype
        alpha = 1.702 if case["dtype"] == "float32" else 1.703125
    return gate * torch.sigmoid(alpha * gate) * (up + case["offset"]) * w[:, None]


def _exact_layer(case, seed):
    x = _inputs(case, seed)
    dt, e, k, t = _dtype(case), case["experts"], case["k"], case["tokens"]
    mx, square = case["fmt"] != "compute", case["fmt"] == "mxfp8_2d"

    def quant(v, kernel=False):
        return _blocks(v, square and kernel) if mx else v

    order = torch.argsort(x["idx"].reshape(-1).long(), stable=True)
    inverse = torch.argsort(order).view(t, k)
    sizes = torch.bincount(x["idx"].reshape(-1).long(), minlength=e).tolist()
    spans, at = [], 0
    for size in sizes:
        spans.append((at, at + size))
        at += size
    expert = torch.repeat_interleave(torch.arange(e, device="cuda"),
                                     torch.tensor(sizes, device="cuda"))

    def rows(a, kernel, transposed):  # each group's rows of a by its kernel, rounded
        y = None
        for g, (lo, hi) in enumerate(spans):
            if hi > lo:
                w = kernel[g].reshape(kernel.shape[1], -1).double()
                w = quant(w, True).T if transposed else quant(w.T.contiguous(), True).T
                part = a[lo:hi] @ w
                y = part.new_empty(a.shape[0], part.shape[1]) if y is None else y
                y[lo:hi] = part
        return _rounded(y, dt)

    def contract(a, b):  # each group's a^T b, both quantized along the rows
        out = torch.empty(e, a.shape[1], b.shape[1], dtype=torch.float64, device="cuda")
        a, b = quant(a.T.contiguous()), quant(b.T.contiguous())
        for g, (lo, hi) in enumerate(spans):
            out[g] = a[:, lo:hi] @ b[:, lo:hi].T
        return out

    def by_expert(v):  # each expert's sum of its rows
        return torch.zeros(e, v.shape[1], dtype=v.dtype, device="cuda").index_add_(0, expert, v)

    xs = x["z"].double()[order // k]
    w = x["weights"].double().reshape(-1)[order]
    act_w = torch.ones_like(w) if case["norm"] else w
    projected = rows(quant(xs), x["up"], False)
    if case["bias"]:
        projected = _rounded(projected + x["up_bias"].double().view(e, -1)[expert], dt)
    h = _rounded(_activation(case, projected, act_w), dt)
    y = rows(quant(h), x["down"], False)
    bias = x["down_bias"].double() if case["bias"] else None

    def normed(y, w, scale):
        v = y if bias is None else y + bias[expert]
        v = v * torch.rsqrt(v.square().mean(-1, keepdim=True) + 1e-6)
        return v * scale * w[:, None]

    if case["norm"]:
        out = _rounded(_rounded(normed(y, w, x["norm_scale"].double()), dt)[inverse].sum(1), dt)
    else:
        out = _rounded(y[inverse].sum(1), dt)
        if bias is not None:
            picked = _rounded(bias[expert] * w[:, None], dt)[inverse].sum(1)
            out = _rounded(out + _rounded(picked, dt), dt)
    if not case["step"]:
        return {"out": out}

    got = {"out": out}
    g = x["dy"].double()[order // k]
    if case["norm"]:
        yv, wv, sv = (v.clone().requires_grad_() for v in (y, w, x["norm_scale"].double()))
        dv, d_w, got["norm_scale"] = torch.autograd.grad(normed(yv, wv, sv), (yv, wv, sv), g)
        g = _rounded(dv, dt)
        if bias is not None:
            got["down_bias"] = by_expert(g)
    elif bias is not None:
        got["down_bias"] = by_expert(_rounded(g * w[:, None], dt))
    dh = rows(quant(g), x["down"], True)
    got["down"] = _rounded(contract(h, g), dt)
    pv, wv = projected.clone().requires_grad_(), act_w.clone().requires_grad_()
    dp, d_act = torch.autograd.grad(_activation(case, pv, wv), (pv, wv), dh)
    dp = _rounded(dp, dt)
    if not case["norm"]:
        d_w = _rounded(d_act, dt)
        if bias is not None:
            d_w = d_w + (g * bias[expert]).sum(-1)
    if case["bias"]:
        got["up_bias"] = by_expert(dp).view(e, -1, 2)
    dx = rows(quant(dp), x["up"], True)
    got["up"] = _rounded(contract(xs, dp), dt).view(e, case["d"], -1, 2)
    got["z"] = _rounded(dx[inverse].sum(1), dt)
    got["weights"] = _rounded(d_w, dt)[inverse]
    return got


def _exact_route(case, seed):
    state = prepare(case, seed)
    logits = state["z"].double() @ state["kernel"].double()
    scores = torch.softmax(logits, -1) if case["router"] == "softmax" else torch.sigmoid(logits)
    choice = scores if state["router_bias"] is None else scores + state["router_bias"].double()
    n = case["groups"]
    if n > 1:  # the best groups by their two best choices
        parts = choice.view(len(choice), n, -1)
        best = torch.topk(parts.topk(2, -1).values.sum(-1), case["top_groups"], -1).indices
        keep = torch.zeros(len(choice), n, dtype=torch.bool, device="cuda").scatter_(1, best, True)
        choice = torch.where(keep[..., None], parts, -torch.inf).view_as(choice)
    idx = torch.topk(choice, case["k"], -1).indices
    w = torch.gather(scores, 1, idx)
    w = _rounded(w / w.sum(-1, keepdim=True), BF16) * case["scaling"]
    return {"idx": None, "weights": _rounded(w, BF16)}


def exact(case, seed):
    if case["kind"] == "layer":
        return _exact_layer(case, seed)
    if case["kind"] == "route":
        return _exact_route(case, seed)
    if case["kind"] == "dispatch":
        state = prepare(case, seed)
        rows = _blocks(state["z"].double())[state["order"].long() // case["k"]]
        return {"packed": None, "rows": _rounded(rows, BF16)}
    return None  # bytes alone
