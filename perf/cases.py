"""The work that users of this framework have it do, as cases to time.

A case is a dict of plain values; `prepare` makes what a program holds before
the call (weights, modules, inputs, a captured graph), `run` is one pass
through the public entry points, `exact` the same result in plain torch at
64 bits.  Block shapes are the configurations of mlx_rs_amd.workloads; the
weights are N(0, 0.02) affine-quantised here in plain torch, x is N(0, 1).
"""
import math

import torch

from __graft_entry__ import load_package

pkg = load_package()
CONFIGS = pkg.workloads.CONFIGS

# most tokens of one call per configuration (prompt chunks)
MAX_T = {"c2": 4096, "c3": 4096, "c4": 2048, "c5": 512, "c6": 2048, "c7": 2048, "c8": 2048}


def listed():
    return [
        # one token of one sequence: the latency of interactive decoding
        {"name": "decode_c2_T1", "kind": "block", "cfg": "c2", "tokens": 1, "graph": False},
        # a small decode batch of the shipped Qwen3.6 layer tail (norm, 8-bit
        # router, shared expert, residual add), replayed from a HIP graph as a
        # serving loop does
        {"name": "tail_c6_T7_graph", "kind": "tail", "cfg": "c6", "tokens": 7, "graph": True},
        # the benchmark's decode batch
        {"name": "decode_c2_T64", "kind": "block", "cfg": "c2", "tokens": 64, "graph": False},
        # the same kind of batch on an unquantised checkpoint (bf16 experts)
        {"name": "decode_c8_T48_bf16", "kind": "block", "cfg": "c8", "tokens": 48, "graph": False},
        # 8-bit experts, wide layer, skewed routing, decode batch
        {"name": "decode_c5_T32_8bit", "kind": "block", "cfg": "c5", "tokens": 32, "graph": False},
        # gemma4's layout (bf16 router, packed GeGLU experts): a large decode
        # batch or a short prompt
        {"name": "gemma_c7_T190", "kind": "block", "cfg": "c7", "tokens": 190, "graph": False},
        # a long prompt under skewed routing
        {"name": "prefill_c3_T4096", "kind": "block", "cfg": "c3", "tokens": 4096, "graph": False},
        # many small experts and a shared expert, a prompt chunk
        {"name": "prefill_c4_T2048", "kind": "block", "cfg": "c4", "tokens": 2048, "graph": False},
        # 8-bit experts, a prompt chunk: the largest weights
        {"name": "prefill_c5_T512_8bit", "kind": "block", "cfg": "c5", "tokens": 512,
         "graph": False},
        # one expert projection as an op (QuantizedSwitchLinear.apply) on a
        # ragged chunk, indices chosen by the caller's own router
        {"name": "gather_qmm_c6_T509", "kind": "gather", "cfg": "c6", "tokens": 509,
         "proj": "up"},
        # converting a checkpoint: one expert bank quantised
        {"name": "quantize_c2_bank", "kind": "quantize", "experts": 128, "rows": 768,
         "cols": 2048, "group": 64, "bits": 4, "f32": False},
        # and read back to bf16
        {"name": "dequantize_c2_bank", "kind": "dequantize", "experts": 128, "rows": 768,
         "cols": 2048, "group": 64, "bits": 4, "f32": False},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choices(["block", "tail", "gather", "quantize", "dequantize"],
                       [9, 3, 2, 1, 1])[0]
    if kind in ("quantize", "dequantize"):
        bits, group = rng.choice([2, 4, 4, 4, 8, 8]), rng.choice([32, 64, 64, 64, 128])
        return {"kind": kind, "experts": _log_int(rng, 1, 128),
                "rows": rng.randint(1, 768), "cols": 128 * rng.randint(1, 16),
                "group": group, "bits": bits, "f32": rng.random() < 0.25}
    if kind == "tail":
        cfg = rng.choice(["c4", "c6", "c8"])
    elif kind == "gather":
        cfg = rng.choice(["c2", "c5", "c6", "c8"])
    else:
        cfg = rng.choice(["c2", "c3", "c4", "c5", "c6", "c7", "c8"])
    case = {"kind": kind, "cfg": cfg, "tokens": _log_int(rng, 1, MAX_T[cfg])}
    if kind == "gather":
        case["proj"] = rng.choice(["up", "down"])
    else:
        case["graph"] = rng.random() < 0.3
    return case


# ------------------------------------------------------------------ inputs
def _device():
    return torch.device("cuda", torch.cuda.current_device())


class _Gen:
    """Seeded normal and uniform tensors, one stream after another."""

    def __init__(self, seed):
        self.dev = _device()
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(seed * 7919 + 17)

    def normal(self, shape, std=1.0, dtype=torch.float32):
        return (torch.randn(shape, generator=self.g, device=self.dev) * std).to(dtype)

    def rand(self, shape):
        return torch.rand(shape, generator=self.g, device=self.dev)


def _quantize(w, group, bits):
    """MLX affine quantisation of w [..., cols] in plain torch: packed codes
    (int32), scales and biases in w's dtype."""
    v = w.float().reshape(w.shape[:-1] + (-1, group))
    hi, lo = v.amax(-1), v.amin(-1)
    bins = float(2 ** bits - 1)
    neg = lo.abs() > hi.abs()
    scale = ((hi - lo) / bins).clamp_min(1e-7)
    scale = torch.where(neg, scale, -scale)
    edge = torch.where(neg, lo, hi)
    q0 = torch.round(edge / scale)
    some = q0 != 0
    scale = torch.where(some, edge / torch.where(some, q0, torch.ones_like(q0)), scale)
    bias = torch.where(some, edge, torch.zeros_like(edge))
    code = torch.round((v - bias[..., None]) / scale[..., None]).clamp_(0, bins).to(torch.int32)
    per = 32 // bits
    code = code.reshape(w.shape[:-1] + (-1, per))
    word = torch.zeros(code.shape[:-1], dtype=torch.int32, device=w.device)
    for k in range(per):
        word |= code[..., k] << (k * bits)
    return word, scale.to(w.dtype), bias.to(w.dtype)


def _dequantize64(t, group, bits):
    """64-bit weights of (codes, scales, biases)."""
    word, s, b = t
    shifts = torch.arange(0, 32, bits, device=word.device, dtype=torch.int32)
    code = ((word[..., None] >> shifts) & (2 ** bits - 1)).double()
    code = code.reshape(s.shape + (group,))
    return (code * s.double()[..., None] + b.double()[..., None]).flatten(-2)


def _bank(g, shape, bits):
    """Expert weights [E, N, K]: a bf16 tensor, or (codes, scales, biases)."""
    if bits == 16:
        out = torch.empty(shape, dtype=torch.bfloat16, device=g.dev)
        for e in range(0, shape[0], 16):
            out[e:e + 16] = g.normal(out[e:e + 16].shape, 0.02, torch.bfloat16)
        return out
    E, N, K = shape
    out = (torch.empty((E, N, K * bits // 32), dtype=torch.int32, device=g.dev),
           torch.empty((E, N, K // 64), dtype=torch.bfloat16, device=g.dev),
           torch.empty((E, N, K // 64), dtype=torch.bfloat16, device=g.dev))
    for e in range(0, E, 16):
        n = min(16, E - e)
        for o, t in zip(out, _quantize(g.normal((n, N, K), 0.02, torch.bfloat16), 64, bits)):
            o[e:e + 16] = t
    return out


def _tensors(case, seed):
    """Every input tensor of a block, tail or gather case."""
    c = CONFIGS[case["cfg"]]
    g = _Gen(seed)
    T = case["tokens"]
    t = {"x": g.normal((T, c.d), 1.0, torch.bfloat16)}
    if case["kind"] == "gather":
        shape = (c.E, c.f, c.d) if case["proj"] == "up" else (c.E, c.d, c.f)
        if case["proj"] == "down":
            t["x"] = g.normal((T, c.f), 1.0, torch.bfloat16)
        t["w"] = _bank(g, shape, c.bits)
        t["idx"] = g.rand((T, c.E)).topk(c.K, dim=1).indices.to(torch.int32)
        return t
    if c.layout == "gemma":
        t["gate"] = g.normal((c.E, c.d), 1.0, torch.bfloat16)
        t["scale"] = torch.ones(c.d, device=g.dev, dtype=torch.bfloat16)
        t["pes"] = (0.5 + g.rand((c.E,))).to(torch.bfloat16)
        t["gate_up"] = _bank(g, (c.E, 2 * c.f, c.d), c.bits)
        t["down"] = _bank(g, (c.E, c.d, c.f), c.bits)
        return t

    def router(rows):
        w = g.normal((rows, c.d), 0.02)
        if c.router_bits == 0:
            return w
        w = w.to(torch.bfloat16)
        return w if c.router_bits == 16 else _quantize(w, 64, c.router_bits)

    t["gate"] = router(c.E)
    t["bias"] = pkg.workloads.zipf_bias(c, g.dev) if c.zipf_alpha else None
    t["gate_proj"] = _bank(g, (c.E, c.f, c.d), c.bits)
    t["up_proj"] = _bank(g, (c.E, c.f, c.d), c.bits)
    t["down"] = _bank(g, (c.E, c.d, c.f), c.bits)
    if c.fs:
        t["shared"] = [_bank(g, s, c.bits) for s in
                       ((1, c.fs, c.d), (1, c.fs, c.d), (1, c.d, c.fs))]
        t["shared_gate"] = router(1)
    if case["kind"] == "tail":
        t["norm"] = (1.0 + g.normal((c.d,), 0.1)).to(torch.bfloat16)
    return t


def _dense_or_quantized(case, seed):
    """The bank of a quantize or dequantize case."""
    g = _Gen(seed)
    dtype = torch.float32 if case["f32"] else torch.bfloat16
    return g.normal((case["experts"], case["rows"], case["cols"]), 0.02, dtype)


# ----------------------------------------------------------------- prepare
def prepare(case, seed):
    nn = pkg.nn
    if case["kind"] == "quantize":
        return {"case": case, "w": _dense_or_quantized(case, seed)}
    if case["kind"] == "dequantize":
        q = _quantize(_dense_or_quantized(case, seed), case["group"], case["bits"])
        return {"case": case, "q": q}
    c = CONFIGS[case["cfg"]]
    t = _tensors(case, seed)

    def switch(w):
        return nn.SwitchLinear(w) if c.bits == 16 else nn.QuantizedSwitchLinear(*w, 64, c.bits)

    def linear(w, bits):
        return nn.Linear(w) if bits == 16 else nn.QuantizedLinear(*w, 64, bits)

    if case["kind"] == "gather":
        # x [T, 1, 1, K] against indices [T, top_k], as SplitSwitchFfn's own
        # projections are applied
        return {"case": case, "mod": switch(t["w"]), "x": t["x"][:, None, None, :],
                "idx": t["idx"]}
    if c.layout == "gemma":
        mod = nn.GemmaMoe(nn.GemmaRouter(t["gate"], t["scale"], t["pes"], c.K),
                          nn.PackedSwitchFfn(switch(t["gate_up"]), switch(t["down"]), "geglu"))
    else:
        def router(w):
            return w if c.router_bits == 0 else linear(w, c.router_bits)
        shared = sgate = None
        if c.fs:
            def one(w):
                return linear(w[0] if c.bits == 16 else tuple(p[0] for p in w), c.bits)
            shared = nn.SwigluMlp(*[one(w) for w in t["shared"]])
            sgate = router(t["shared_gate"])
        mod = nn.Qwen35MoeBlock(
            router(t["gate"]),
            nn.SplitSwitchFfn(switch(t["gate_proj"]), switch(t["up_proj"]), switch(t["down"])),
            c.K, shared, sgate, t["bias"])
    st = {"case": case, "mod": mod, "x": t["x"],
          "norm": nn.RmsNorm(t["norm"]) if case["kind"] == "tail" else None}
    if case["graph"]:
        _call(st)  # first use outside the capture
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            st["out"] = _call(st)
    return st


def _call(st):
    m = st["mod"]
    y = m.forward_residual(st["x"], st["norm"]) if st["norm"] is not None else m(st["x"])
    return {"out": y, "indices": m.last_indices, "weights": m.last_weights}


def run(state):
    case = state["case"]
    if case["kind"] == "quantize":
        return pkg.ops.quantize(state["w"], case["group"], case["bits"])
    if case["kind"] == "dequantize":
        return pkg.ops.dequantize(*state["q"], case["group"], case["bits"])
    if case["kind"] == "gather":
        return state["mod"].apply(state["x"], state["idx"])
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _call(state)


# -------------------------------------------------------- work, tolerance
def _distinct(c, T):
    """Expected distinct experts of T tokens: uniform routing, or Zipf."""
    p = [1.0] * c.E
    if c.zipf_alpha:
        p = [(r + 1) ** -c.zipf_alpha for r in range(c.E)]
    s = sum(p)
    return sum(1.0 - (1.0 - min(1.0, c.K * q / s)) ** T for q in p)


def work(case):
    if case["kind"] in ("quantize", "dequantize"):
        n = case["experts"] * case["rows"] * case["cols"]
        e = 4 if case["f32"] else 2
        return {"bytes": int(n * (e + case["bits"] / 8 + 2 * e / case["group"])), "flops": 4 * n}
    c = CONFIGS[case["cfg"]]
    T = case["tokens"]
    per_w = 2.0 if c.bits == 16 else c.bits / 8 + 4 / 64
    U = _distinct(c, T)
    if case["kind"] == "gather":
        k, n = (c.d, c.f) if case["proj"] == "up" else (c.f, c.d)
        U = c.E * (1 - (1 - c.K / c.E) ** T)
        return {"bytes": int(U * c.f * c.d * per_w + T * k * 2 + T * c.K * (n * 2 + 4)),
                "flops": 2 * T * c.K * c.f * c.d}
    per_r = 2 if c.router_bits == 16 else c.router_bits / 8 + 4 / 64 if c.router_bits else 4
    b = U * 3 * c.f * c.d * per_w + c.E * c.d * per_r
    fl = 6 * T * c.K * c.f * c.d + 2 * T * c.d * c.E
    if c.fs:
        b += 3 * c.fs * c.d * per_w + c.d * per_r
        fl += 6 * T * c.fs * c.d + 2 * T * c.d
    b += T * c.d * 2 + T * c.d * (2 if c.router_bits else 4) + T * c.K * 8
    return {"bytes": int(b), "flops": int(fl)}


def tolerance(case):
    # codes and bf16 scales are bytes; dequantised values are rounded once
    if case["kind"] in ("quantize", "dequantize"):
        return "exact"
    # one bf16 product row: f32 sums, one rounding (bf16 weights when tiled)
    if case["kind"] == "gather":
        return {"rel": 7e-3}
    # a block rounds its activations and expert rows to bf16 on the way.  The
    # routing is computed in f32 in a fixed order: ids differ only at ties.
    return {"rel": 1.5e-2, "differ": 1e-3}


# ------------------------------------------------------------------- exact
def _rb(v):
    """Rounded to bf16, kept in 64 bits."""
    return v.to(torch.bfloat16).double()


def _w64(w, e, bits):
    return w[e].double() if bits == 16 else _dequantize64(tuple(p[e] for p in w), 64, bits)


def _router64(c, w):
    if c.router_bits in (4, 8):
        return _dequantize64(w, 64, c.router_bits)
    return w.double()


def _silu(v):
    return v / (1.0 + torch.exp(-v))


def _geglu(v):
    # gelu_approximate with the constants as the checkpoint's bf16 holds them
    k, s = 0.044677734375, 0.796875
    return 0.5 * v * (1.0 + torch.tanh(s * (v + k * v ** 3)))


def _topk(score, K):
    """Largest K, ties to the lower index."""
    order = torch.sort(score, dim=1, descending=True, stable=True)
    return order.values[:, :K], order.indices[:, :K]


def exact(case, seed):
    if case["kind"] == "quantize":
        w = _dense_or_quantized(case, seed)
        _, s, b = _quantize64(w, case["group"], case["bits"])
        return (None, s, b)
    if case["kind"] == "dequantize":
        q = _quantize(_dense_or_quantized(case, seed), case["group"], case["bits"])
        return _dequantize64(q, case["group"], case["bits"])
    c = CONFIGS[case["cfg"]]
    t = _tensors(case, seed)
    x = t["x"].double()
    T = case["tokens"]
    if case["kind"] == "gather":
        idx = t["idx"].long()
        n = c.f if case["proj"] == "up" else c.d
        y = torch.empty((T, c.K, 1, n), dtype=torch.float64, device=x.device)
        for e in torch.unique(idx).tolist():
            r, k = (idx == e).nonzero(as_tuple=True)
            y[r, k, 0] = x[r] @ _w64(t["w"], e, c.bits).t()
        return y
    h = x
    if case["kind"] == "tail" or c.layout == "gemma":
        # the norm's output is a bf16 tensor that router and experts read;
        # gemma4's experts take the router's input as it was
        wn = (t["norm"] if case["kind"] == "tail" else
              t["scale"] * torch.tensor(c.d ** -0.5, dtype=torch.bfloat16, device=x.device)).double()
        r = torch.rsqrt((x * x).mean(1, keepdim=True) + 1e-6)
        h = _rb(wn * _rb(x * r))
        if case["kind"] == "tail":
            x = h
    logits = h @ _router64(c, t["gate"]).t()
    if c.layout == "gemma":
        s, idx = _topk(_rb(logits), c.K)
        p = _rb(torch.softmax(s - s[:, :1], 1))
        w = _rb(p * t["pes"].double()[idx])
    elif c.router_bits:
        # the bf16 chain: logits, probabilities and weights are bf16 tensors
        p, idx = _topk(_rb(torch.softmax(_rb(logits), 1)), c.K)
        w = _rb(p / _rb(p.sum(1, keepdim=True)))
    else:
        if t["bias"] is not None:
            logits = logits + t["bias"].double()
        p, idx = _topk(torch.softmax(logits, 1), c.K)
        w = p / p.sum(1, keepdim=True)
    out = torch.zeros_like(x)
    for e in torch.unique(idx).tolist():
        r, k = (idx == e).nonzero(as_tuple=True)
        if c.layout == "gemma":
            gu = x[r] @ _w64(t["gate_up"], e, c.bits).t()
            a = _geglu(gu[:, :c.f]) * gu[:, c.f:]
        else:
            a = (_silu(x[r] @ _w64(t["gate_proj"], e, c.bits).t()) *
                 (x[r] @ _w64(t["up_proj"], e, c.bits).t()))
        out.index_add_(0, r, w[r, k][:, None] * (a @ _w64(t["down"], e, c.bits).t()))
    if c.layout != "gemma" and c.fs:
        g, u, d = (_w64(m, 0, c.bits) for m in t["shared"])
        sl = x @ _router64(c, t["shared_gate"]).t()
        out = out + torch.sigmoid(sl) * ((_silu(x @ g.t()) * (x @ u.t())) @ d.t())
    if case["kind"] == "tail":
        out = out + t["x"].double()
    return {"out": out, "indices": None, "weights": w}


def _quantize64(w, group, bits):
    v = w.double().reshape(w.shape[:-1] + (-1, group))
    hi, lo = v.amax(-1), v.amin(-1)
    neg = lo.abs() > hi.abs()
    scale = ((hi - lo) / (2 ** bits - 1)).clamp_min(1e-7)
    scale = torch.where(neg, scale, -scale)
    edge = torch.where(neg, lo, hi)
    q0 = torch.round(edge / scale)
    some = q0 != 0
    return (None, torch.where(some, edge / torch.where(some, q0, torch.ones_like(q0)), scale),
            torch.where(some, edge, torch.zeros_like(edge)))
