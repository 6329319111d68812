"""Performance cases of the op pack: what a serving program calls, on one GPU.

Five kinds of work, each through the package's public entry points:

* ``linear``   one projection of a model: the fp8-weight GEMV / GEMM ops over
               the projection's weights in ``layers`` consecutive layers, as a
               decode step or a prefill chunk calls them (so that, as in a
               model, a call does not find its weights in the caches unless
               the model is tiny);
* ``attn_in``  add+RMSNorm (+ per-token e4m3 quantisation) -> QKV projection
               -> QK-norm + RoPE, per layer;
* ``mlp``      add+RMSNorm (+ quantisation) -> gate/up projection with
               gelu_and_mul -> (quantisation ->) down projection, per layer;
* ``decode``   a whole decode step over a stack of decoder layers, captured
               once in a HIP graph and replayed on new inputs;
* ``norm``     the in-place batched add+RMSNorm.

Sizes are those of the benchmark configurations (hidden 3072, 4096, 5120, MLP
14336 and 24576, QKV 6144), of the reference's own test shapes (hidden 2560,
K = 10240 and 10752) and generic ones.  Weights are N(0, 0.02) quantised per
row or per tensor, activations N(0, 1), norm weights 1 + N(0, 0.1).
"""

import math

import torch

import esimd_learning_amd

_ops = esimd_learning_amd.ops()

DEV = "cuda"
EPS = 1e-6
THETA = 10000.0
FP8_MAX = {"e4m3": 448.0, "e5m2": 57344.0}
FP8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
IO = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _linear(m, k, n, io="fp16", fmt="e4m3", scale="channel", layers=1):
    return {"kind": "linear", "m": m, "k": k, "n": n, "io": io, "fmt": fmt, "scale": scale, "layers": layers}


def _attn_in(m, h, nq, nk, hd, io="fp16", act="fp8", layers=1):
    return {"kind": "attn_in", "m": m, "h": h, "nq": nq, "nk": nk, "hd": hd, "io": io, "act": act, "layers": layers}


def _mlp(m, h, d, io="fp16", act="fp8", layers=1):
    return {"kind": "mlp", "m": m, "h": h, "d": d, "io": io, "act": act, "layers": layers}


def _decode(m, hidden, heads, hd, mlp, layers):
    return {"kind": "decode", "m": m, "h": hidden, "heads": heads, "hd": hd, "d": mlp, "layers": layers}


def _norm(m, h, io="fp16"):
    return {"kind": "norm", "m": m, "h": h, "io": io}


def listed():
    return [
        # one token through a small model's projection: launch latency
        dict(_linear(1, 2048, 2560), name="gemv_m1_small"),
        # one token, the benchmark's headline projection (one request being decoded)
        dict(_linear(1, 4096, 14336, layers=4), name="gemv_m1_headline"),
        # four requests, a long-K down projection with e5m2 weights and one scale per tensor
        dict(_linear(4, 10240, 2560, fmt="e5m2", scale="tensor", layers=8), name="gemv_m4_down_e5m2"),
        # eight requests in bf16 through the gate/up matrix of a hidden-2560 model
        dict(_linear(8, 2560, 20480, io="bf16", scale="tensor", layers=4), name="gemv_m8_bf16"),
        # sixteen requests, fused QKV matrix
        dict(_linear(16, 4096, 6144, layers=8), name="gemv_m16_qkv"),
        # a larger decode batch (or speculative tokens) through the GEMM op
        dict(_linear(48, 4096, 6144, scale="tensor", layers=8), name="gemm_m48"),
        # a ragged prefill chunk in bf16
        dict(_linear(333, 2560, 10752, io="bf16", scale="tensor", layers=4), name="gemm_m333_bf16"),
        # a long prompt, 16-bit activations
        dict(_linear(4096, 4096, 6144, scale="tensor"), name="gemm_m4096"),
        # a decode batch with fp8 hand-offs: norm+quant, QKV, QK-norm+RoPE
        dict(_attn_in(64, 5120, 32, 8, 128, layers=4), name="attn_in_m64_fp8"),
        # prefill of an MLP with fp8 hand-offs (the largest)
        dict(_mlp(2048, 4096, 14336), name="mlp_m2048_fp8"),
        # a whole decode step, four requests, graph-replayed
        dict(_decode(4, 3072, 16, 256, 24576, 4), name="decode_m4"),
        # the residual add and norm of a prefill chunk
        dict(_norm(2048, 5120, io="bf16"), name="norm_m2048_bf16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _rows(rng):
    """Tokens of a call: half decode batches, the rest mixed batches and prompts."""
    part = rng.random()
    return _log_int(rng, 1, 16) if part < 0.5 else (_log_int(rng, 17, 128) if part < 0.75 else _log_int(rng, 129, 4096))


def _layers(weight_bytes, flops):
    """Layers of a call: about 100 MB of weights where that stays a short call."""
    return max(1, min(8, int(100e6 / weight_bytes), int(1e11 / flops)))


def draw(rng):
    kind = rng.choices(["linear", "attn_in", "mlp", "decode", "norm"], [50, 15, 15, 8, 12])[0]
    io = rng.choice(["fp16", "fp16", "bf16"])
    if kind == "linear":
        m = _rows(rng)
        # model widths: multiples of 256, sometimes only of 64; any number of outputs
        unit = rng.choice([256, 256, 64])
        k = unit * max(1, _log_int(rng, 1024, 16384) // unit)
        n = _log_int(rng, 128, 32768)
        if rng.random() < 0.75:
            n = 128 * max(1, n // 128)
        while 2.0 * m * n * k > 4e11:
            m = max(1, m // 2)
        return _linear(m, k, n, io=io, fmt=rng.choice(["e4m3", "e4m3", "e4m3", "e5m2"]),
                       scale=rng.choice(["channel", "tensor"]), layers=_layers(n * k, 2.0 * m * n * k))
    if kind == "norm":
        return _norm(_log_int(rng, 1, 8192), 64 * rng.choice([24, 32, 40, 48, 56, 64, 80, 96, 112, 128]), io=io)
    if kind == "decode":
        h, heads, hd, d = rng.choice([(3072, 16, 256, 24576), (2048, 8, 256, 16384), (4096, 32, 128, 14336),
                                      (2560, 10, 256, 10240)])
        return _decode(_log_int(rng, 1, 16), h, heads, hd, d, rng.choice([1, 2, 3, 4]))
    m = _rows(rng)
    act = rng.choice(["fp8", "fp8", "io"])
    h = 256 * rng.choice([8, 10, 12, 16, 20, 28, 32])
    if kind == "attn_in":
        hd = rng.choice([64, 128, 128, 256])
        nq = rng.choice([8, 16, 28, 32])
        nk = rng.choice([v for v in (1, 2, 4, 8, nq) if nq % v == 0])
        n = (nq + 2 * nk) * hd
        return _attn_in(m, h, nq, nk, hd, io=io, act=act, layers=_layers(n * h, 2.0 * m * n * h))
    d = 256 * rng.choice([16, 24, 32, 40, 56, 64])
    while 6.0 * m * h * d > 6e11:
        m //= 2
    return _mlp(m, h, d, io=io, act=act, layers=_layers(3 * h * d, 6.0 * m * h * d))


# ---- inputs (plain torch) ---------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _weight(g, n, k, fmt="e4m3", scale="channel"):
    w = torch.randn(n, k, device=DEV, generator=g).mul_(0.02)
    if scale == "channel":
        s = w.abs().amax(dim=1) / FP8_MAX[fmt]
        w.div_(s[:, None])
    else:
        s = w.abs().amax().reshape(1) / FP8_MAX[fmt]
        w.div_(s)
    return w.clamp_(-FP8_MAX[fmt], FP8_MAX[fmt]).to(FP8[fmt]), s


def _act(g, m, h, io):
    return torch.randn(m, h, device=DEV, generator=g).to(IO[io])


def _norm_weight(g, h, io):
    return (1.0 + 0.1 * torch.randn(h, device=DEV, generator=g)).to(IO[io])


def _positions(g, m):
    return torch.randint(0, 8192, (m,), device=DEV, generator=g, dtype=torch.int64)


def _inputs(c, seed):
    g, kind, m = _gen(seed), c["kind"], c["m"]
    if kind == "linear":
        return {"x": _act(g, m, c["k"], c["io"]),
                "w": [_weight(g, c["n"], c["k"], c["fmt"], c["scale"]) for _ in range(c["layers"])]}
    if kind == "norm":
        return {"h": _act(g, m, c["h"], c["io"]), "r": _act(g, m, c["h"], c["io"]),
                "g": _norm_weight(g, c["h"], c["io"])}
    if kind == "attn_in":
        n = (c["nq"] + 2 * c["nk"]) * c["hd"]
        return {"h": _act(g, m, c["h"], c["io"]), "r": _act(g, m, c["h"], c["io"]), "pos": _positions(g, m),
                "layers": [{"g": _norm_weight(g, c["h"], c["io"]), "w": _weight(g, n, c["h"]),
                            "qw": _norm_weight(g, c["hd"], c["io"]), "kw": _norm_weight(g, c["hd"], c["io"])}
                           for _ in range(c["layers"])]}
    if kind == "mlp":
        return {"h": _act(g, m, c["h"], c["io"]), "r": _act(g, m, c["h"], c["io"]),
                "layers": [{"g": _norm_weight(g, c["h"], c["io"]), "wgu": _weight(g, 2 * c["d"], c["h"]),
                            "wd": _weight(g, c["h"], c["d"])} for _ in range(c["layers"])]}
    nq = c["heads"] * c["hd"]
    layers = []
    for _ in range(c["layers"]):
        p = {"hidden": c["h"], "n_q": c["heads"], "n_kv": c["heads"], "head_dim": c["hd"], "mlp": c["d"],
             "eps": EPS, "theta": THETA}
        for name, n, k in (("qkv", 3 * nq, c["h"]), ("o", c["h"], nq), ("gu", 2 * c["d"], c["h"]),
                           ("d", c["h"], c["d"])):
            p["W" + name], p["s" + name] = _weight(g, n, k)
        p["w_in"], p["w_post"] = _norm_weight(g, c["h"], "fp16"), _norm_weight(g, c["h"], "fp16")
        p["qw"], p["kw"] = _norm_weight(g, c["hd"], "fp16"), _norm_weight(g, c["hd"], "fp16")
        layers.append(p)
    return {"h": _act(g, m, c["h"], "fp16"), "r": _act(g, m, c["h"], "fp16"), "pos": _positions(g, m),
            "layers": layers}


# ---- the calls ---------------------------------------------------------------


def prepare(case, seed):
    s = dict(_inputs(case, seed), case=case)
    kind, m = case["kind"], case["m"]
    new = lambda n, dt: torch.empty(m, n, dtype=dt, device=DEV)  # noqa: E731
    if kind == "linear":
        s["y"] = [new(case["n"], IO[case["io"]]) for _ in s["w"]]
    elif kind in ("attn_in", "mlp"):
        dt, h = IO[case["io"]], case["h"]
        for layer in s["layers"]:
            layer["r_out"] = new(h, dt)
            if kind == "attn_in":
                layer["qkv"] = new(layer["w"][0].shape[0], dt)
            else:
                layer["act"], layer["out"] = new(case["d"], dt), new(h, dt)
            if case["act"] == "fp8":
                layer["q8"], layer["s8"] = new(h, torch.float8_e4m3fn), torch.empty(m, device=DEV)
                if kind == "mlp":
                    layer["a8"], layer["as8"] = new(case["d"], torch.float8_e4m3fn), torch.empty(m, device=DEV)
    elif kind == "decode":
        from esimd_learning_amd.layer import GemmaDecodeLayer, capture_forward, forward
        s["stack"] = [GemmaDecodeLayer(p, m, DEV) for p in s.pop("layers")]
        s["hidden"], s["residual"] = s["h"].clone(), s["r"].clone()
        forward(s["stack"], s["hidden"], s["residual"], s["pos"])
        s["graph"] = capture_forward(s["stack"], s["hidden"], s["residual"], s["pos"])
    return s


def _run_linear(s, c):
    m, n, k, x = c["m"], c["n"], c["k"], s["x"]
    for (w, sc), y in zip(s["w"], s["y"]):
        if c["scale"] == "channel":
            _ops.esimd_gemv_fp8_pern(x, w, sc, y, n, k)
        elif m <= 16:
            _ops.esimd_gemv_fp8_pert(x, w, sc, y)
        else:
            _ops.esimd_gemm_fp8_pert(x, w, sc, y)
    return s["y"]


def _run_attn_in(s, c):
    nq, nk = c["nq"] * c["hd"], c["nk"] * c["hd"]
    outs = []
    for p in s["layers"]:
        w, sc = p["w"]
        if c["act"] == "fp8":
            _ops.esimd_fused_add_rms_norm_quant_gemv_fp8(s["h"], s["r"], p["g"], EPS, p["r_out"], p["q8"], p["s8"],
                                                         w, sc, p["qkv"])
        else:
            _ops.esimd_fused_add_rms_norm_gemv_fp8(s["h"], s["r"], p["g"], EPS, p["r_out"], w, sc, p["qkv"])
        _ops.esimd_qk_norm_rope(p["qkv"][:, :nq], p["qkv"][:, nq:nq + nk], p["qw"], p["kw"], s["pos"], EPS, THETA,
                                True)
        outs.append({n: p[n] for n in ("r_out", "q8", "s8", "qkv") if n in p})
    return outs


def _run_mlp(s, c):
    outs = []
    for p in s["layers"]:
        (wgu, sgu), (wd, sd) = p["wgu"], p["wd"]
        if c["act"] == "fp8":
            _ops.esimd_fused_add_rms_norm_quant_gemv_fp8(s["h"], s["r"], p["g"], EPS, p["r_out"], p["q8"], p["s8"],
                                                         wgu, sgu, p["act"], True)
            _ops.esimd_per_token_quant_fp8(p["act"], p["a8"], p["as8"])
            _ops.esimd_gemm_fp8_a8w8(p["a8"], p["as8"], wd, sd, p["out"])
        else:
            _ops.esimd_fused_add_rms_norm_gemv_fp8(s["h"], s["r"], p["g"], EPS, p["r_out"], wgu, sgu, p["act"], True)
            _ops.esimd_gemv_fp8_pern(p["act"], wd, sd, p["out"], c["h"], c["d"])
        outs.append({n: p[n] for n in ("r_out", "q8", "s8", "act", "out") if n in p})
    return outs


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "linear":
        return _run_linear(state, c)
    if kind == "attn_in":
        return _run_attn_in(state, c)
    if kind == "mlp":
        return _run_mlp(state, c)
    if kind == "norm":
        _ops.esimd_fused_add_rms_norm_batched(state["h"], state["r"], state["g"], EPS)
        return {"hidden": state["h"], "residual": state["r"]}
    # the step's inputs go into the graph's own buffers, which it updates
    state["hidden"].copy_(state["h"])
    state["residual"].copy_(state["r"])
    state["graph"].replay()
    return {"out": state["stack"][-1].out, "residual": state["residual"]}


def work(case):
    c, m = case, case["m"]
    if c["kind"] == "linear":
        n, k = c["n"], c["k"]
        per = n * k + 2 * m * n + (4 * n if c["scale"] == "channel" else 4)
        return {"bytes": c["layers"] * per + 2 * m * k, "flops": c["layers"] * 2.0 * m * n * k}
    h = c["h"]
    if c["kind"] == "norm":
        return {"bytes": 8 * m * h + 2 * h, "flops": 8.0 * m * h}
    if c["kind"] == "attn_in":
        n = (c["nq"] + 2 * c["nk"]) * c["hd"]
        per = n * h + 4 * n + 2 * h + 2 * m * h + 2 * m * n + (m * h + 4 * m if c["act"] == "fp8" else 0)
        return {"bytes": c["layers"] * per + 4 * m * h + 8 * m, "flops": c["layers"] * 2.0 * m * n * h}
    if c["kind"] == "mlp":
        d = c["d"]
        per = 3 * d * h + 8 * d + 6 * h + 2 * m * h + 2 * m * d + 2 * m * h + (m * h + m * d + 8 * m if c["act"] == "fp8" else 0)
        return {"bytes": c["layers"] * per + 4 * m * h, "flops": c["layers"] * 6.0 * m * d * h}
    nq, d = c["heads"] * c["hd"], c["d"]
    w = 4 * nq * h + 3 * d * h
    return {"bytes": c["layers"] * (w + 4 * (3 * nq + 2 * h + 2 * d)) + 8 * m * h, "flops": c["layers"] * 2.0 * m * w}


def tolerance(case):
    """About four times the distance from 64-bit arithmetic that was measured:
    the last rounding to the 16-bit type (fp16 2.1e-4, bf16 1.7e-3), plus, where
    e4m3 codes are made on the way, codes that fall on the other side of a
    rounding boundary (fp16 MLP output 2.5e-3), and in the whole step the
    roundings between its ops (1.9e-3)."""
    bf16 = case.get("io") == "bf16"
    if case["kind"] in ("linear", "norm"):
        return {"rel": 7e-3 if bf16 else 9e-4, "max": 4e-2 if bf16 else 6e-3}
    if case["kind"] == "decode":
        return {"rel": 8e-3, "max": 8e-2}
    if case["kind"] == "mlp" and case["act"] == "fp8":
        return {"rel": 1.5e-2 if bf16 else 1e-2, "max": 0.3}
    # (a code off by one step is an eighth of its value)
    return {"rel": 8e-3 if bf16 else 2e-3, "max": 0.3 if case["act"] == "fp8" else 8e-2}


# ---- the same in 64 bits, plain torch ----------------------------------------


def _f64(t):
    return t.float().double()


def _matmul(x, w):
    """x [m, k] (64-bit) times the dequantised weight's transpose."""
    w8, s = w
    return (x @ _f64(w8).t()) * s.double()


def _add_norm(h, r, g, io):
    """The op's definition: the sum is stored rounded, its squares taken before."""
    a = _f64(h) + _f64(r)
    r_new = a.to(IO[io])
    inv = torch.rsqrt((a * a).mean(-1, keepdim=True) + EPS)
    return r_new, _f64(r_new) * inv * _f64(g)


def _quant(x):
    s = (x.abs().amax(-1) / 448.0).clamp_min(1.0 / (448.0 * 512.0))
    return (x / s[:, None]).clamp(-448.0, 448.0).float().to(torch.float8_e4m3fn), s


def _gelu(u):
    return 0.5 * u * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (u + 0.044715 * u ** 3)))


def _rope(x, w, pos, hd, io):
    """Per-head RMSNorm (its output rounded to io, if given), then the rotation."""
    m = x.shape[0]
    v = x.reshape(m, -1, hd)
    v = v * torch.rsqrt((v * v).mean(-1, keepdim=True) + EPS) * _f64(w)
    if io:
        v = _f64(v.to(IO[io]))
    half = hd // 2
    freq = THETA ** (-torch.arange(half, device=DEV, dtype=torch.float64) * 2.0 / hd)
    ang = (pos.double()[:, None] * freq)[:, None, :]
    cos, sin = torch.cos(ang), torch.sin(ang)
    a, b = v[..., :half], v[..., half:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1).reshape(m, -1)


def exact(case, seed):
    c, i = case, _inputs(case, seed)
    kind = c["kind"]
    if kind == "linear":
        return [_matmul(_f64(i["x"]), w) for w in i["w"]]
    if kind == "norm":
        r, x = _add_norm(i["h"], i["r"], i["g"], c["io"])
        return {"hidden": x, "residual": _f64(r)}
    if kind in ("attn_in", "mlp"):
        io, outs = c["io"], []
        rnd = lambda t: _f64(t.to(IO[io]))  # noqa: E731
        for p in i["layers"]:
            r, x = _add_norm(i["h"], i["r"], p["g"], io)
            o, x, sx = {"r_out": _f64(r)}, rnd(x), 1.0
            if c["act"] == "fp8":
                q, s = _quant(x)
                o["q8"], o["s8"], x, sx = _f64(q), s, _f64(q), s[:, None]
            if kind == "attn_in":
                y = rnd(_matmul(x, p["w"]) * sx)
                nq, nk = c["nq"] * c["hd"], c["nk"] * c["hd"]
                o["qkv"] = torch.cat([_rope(y[:, :nq], p["qw"], i["pos"], c["hd"], io),
                                      _rope(y[:, nq:nq + nk], p["kw"], i["pos"], c["hd"], io), y[:, nq + nk:]], 1)
            else:
                y = rnd(_matmul(x, p["wgu"]) * sx)
                a = rnd(_gelu(y[:, :c["d"]]) * y[:, c["d"]:])
                o["act"] = a
                if c["act"] == "fp8":
                    q, s = _quant(a)
                    o["out"] = _matmul(_f64(q), p["wd"]) * s[:, None]
                else:
                    o["out"] = _matmul(a, p["wd"])
            outs.append(o)
        return outs
    h, r = _f64(i["h"]), _f64(i["r"])
    for p in i["layers"]:
        norm = lambda v, w: v * torch.rsqrt((v * v).mean(-1, keepdim=True) + EPS) * _f64(w)  # noqa: E731
        r = r + h
        qkv = _matmul(norm(r, p["w_in"]), (p["Wqkv"], p["sqkv"]))
        q = _rope(qkv[:, :c["heads"] * c["hd"]], p["qw"], i["pos"], c["hd"], None)
        r = r + _matmul(q, (p["Wo"], p["so"]))
        gu = _matmul(norm(r, p["w_post"]), (p["Wgu"], p["sgu"]))
        h = _matmul(_gelu(gu[:, :c["d"]]) * gu[:, c["d"]:], (p["Wd"], p["sd"]))
    return {"out": h, "residual": r}
