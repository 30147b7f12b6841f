"""The workloads this framework's speed is measured on.

Each case is one call (or one recorded graph of calls) through the public
C ABI of libvai_amd.so, as a Python host makes them with vai_amd._capi: the
argument struct is filled once, weights are packed once where the library has
a packed form, the workspace is sized by the library and kept, and a pass is
the launch. Buffers are torch tensors on the GPU; launches go to torch's
current stream.

  linear     the Linear node: decode (M <= 8), prompts, prefill; fp16 weights
             with fp16 or fp32 activations (fp32 is the engine's default
             between nodes), fp32 weights; bias, residual, activation, gate.
  attention  the Attention node: prefill (causal, windows, GQA) and decode
             over the KV cache.
  scores     the AttentionScores node.
  conv       the Convolution node: 3x3 and 1x1, stride 1 and 2, NCHW.
  decoder    one decode step of a small transformer, recorded as a HIP graph
             and replayed (what a NeuralNet does with its nodes' launches).
"""
import ctypes
import math

import torch

from vai_amd import _capi as capi

TORCH = {"f32": torch.float32, "f16": torch.float16}
BYTES = {"f32": 4, "f16": 2}


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # One token through a large-model up projection (bench.py's config 2): a
        # decode loop's commonest call, bound by reading the weight once.
        _linear("decode_m1", 1, 2048, 8192),
        # A few sequences decoded together through the fused gate/up projection.
        _linear("decode_gate_up_m4", 4, 2048, 16384, gated=True, out="f16"),
        # A short chat prompt through a query/key/value projection, odd length.
        _linear("prompt_qkv_m61", 61, 3072, 5120, bias=True, out="f16"),
        # A prompt in the engine's default dtypes (fp16 weights, fp32 between
        # nodes) through an attention output projection with its residual.
        _linear("prompt_default_dtypes_m500", 500, 2048, 2048, x="f32", residual=True),
        # A long prompt's gate/up projection (config 3).
        _linear("prefill_gate_up_m2048", 2048, 3072, 16384, gated=True),
        # The GPT-2 MLP in fp32 (config 1).
        _linear("gpt2_c_fc_f32", 128, 768, 3072, x="f32", w="f32", bias=True, act="GELU_TANH"),
        # A long prompt's attention, grouped query heads.
        _attention("attention_prefill_t4096", 24, 8, 128, 4096),
        # One token against a KV cache: the attention of every decode step.
        _attention("attention_decode_cache", 32, 8, 64, 1, cache=4096, count=3000),
        # The score matmul alone (config 4).
        {"name": "scores_causal_t1024", "op": "scores", "hq": 8, "hkv": 8, "d": 256, "tq": 1024, "tkv": 1024,
         "x": "f16", "span": 0},
        # YOLOX-s: a body convolution (config 5) and the first downsample of a
        # 640-pixel image, whose rows are the widest in the network.
        _conv("conv3x3_80", 128, 128, 80, 80, 3, 1),
        _conv("conv3x3_s2_320", 32, 64, 320, 320, 3, 2, out="f16"),
        # A whole decode step: many small launches in one recorded graph.
        {"name": "decoder_step", "op": "decoder", "layers": 4, "dim": 2048, "hq": 32, "hkv": 8, "d": 64,
         "ffn": 8192, "vocab": 8192, "cache": 2048, "count": 1200},
    ]


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    kind = rng.choice(("decode", "decode", "prompt", "prompt", "prompt", "f32", "prefill_attention",
                       "prefill_attention", "decode_attention", "decode_attention", "scores", "conv", "conv", "conv",
                       "decoder"))
    if kind == "decode":      # 1-8 rows, any width; the engine's and fp16 activations; gated or not
        k, gated = _size(rng, 512, 8192), rng.random() < 0.3
        n = _size(rng, 512, min(65536, (1 << 27) // k))
        return _linear(None, rng.randint(1, 8), k, n + n % 2 if gated else n, x=rng.choice(("f16", "f32")),
                       out=rng.choice(("f32", "f16")), gated=gated, bias=rng.random() < 0.5,
                       act="NONE" if gated else rng.choice(("NONE", "GELU_TANH", "SILU")))
    if kind == "prompt":      # 9-4096 rows against fp16 weights
        k, gated = _size(rng, 512, 8192), rng.random() < 0.3
        n = _size(rng, 512, 16384)
        m = _log(rng, 9, max(9, min(4096, int(1.5e10 / (2 * k * n)))))
        return _linear(None, m, k, n + n % 2 if gated else n, x=rng.choice(("f16", "f16", "f32")),
                       out=rng.choice(("f32", "f16")), gated=gated, bias=rng.random() < 0.5,
                       residual=not gated and rng.random() < 0.5,
                       act="NONE" if gated else rng.choice(("NONE", "GELU_TANH", "SILU")))
    if kind == "f32":         # fp32 weights, GPT-2 sizes and larger
        k = _size(rng, 512, 3072)
        n = _size(rng, 512, 4096)
        return _linear(None, _log(rng, 1, min(1024, int(6e9 / (2 * k * n)))), k, n, x="f32", w="f32",
                       bias=rng.random() < 0.7, residual=rng.random() < 0.3, act=rng.choice(("NONE", "GELU_TANH")))
    if kind == "prefill_attention":
        hkv = rng.choice((1, 2, 4, 8, 12))
        hq = hkv * rng.choice((1, 1, 2, 4))
        d, t = rng.choice((64, 64, 72, 80, 128, 128, 256)), _log(rng, 33, 4096)
        while 4 * d * hq * t * t > 1e11:
            t = t * 3 // 4
        return _attention(None, hq, hkv, d, t, x=rng.choice(("f16", "f16", "f32")), out=rng.choice(("f16", "f32")),
                          causal=rng.random() < 0.8, span=rng.choice((0, 0, 0, 512)))
    if kind == "decode_attention":
        hkv = rng.choice((1, 2, 4, 8, 12))
        cache = 256 * _log(rng, 1, 64)
        new = rng.choice((1, 1, 1, 1, 4, 16))
        return _attention(None, hkv * rng.choice((1, 2, 4, 8)), hkv, rng.choice((64, 128, 256)), new, cache=cache,
                          count=min(cache - new, _log(rng, 16, 16000)), x=rng.choice(("f16", "f16", "f32")),
                          kv=rng.choice(("f16", "f16", "f16", "f32")), out=rng.choice(("f16", "f32")),
                          span=rng.choice((0, 0, 512)))
    if kind == "scores":
        hkv, tq = rng.choice((1, 4, 8)), _log(rng, 16, 2048)
        tkv = tq if rng.random() < 0.7 else min(4096, tq + _log(rng, 1, 2048))
        hq = hkv * rng.choice((1, 2, 3))
        while hq * tq * tkv > 5e7:
            tq, tkv = tq // 2, tkv // 2
        return {"op": "scores", "hq": hq, "hkv": hkv, "d": rng.choice((64, 72, 128, 256)), "tq": tq,
                "tkv": tkv, "x": rng.choice(("f16", "f16", "f16", "f32")), "span": rng.choice((0, 0, 256))}
    if kind == "conv":        # the stages of an image network: wide and few channels to narrow and many
        w = rng.choice((20, 40, 52, 80, 104, 160, 208, 320, 333))
        h = w if rng.random() < 0.6 else max(8, w - rng.randint(1, w // 2))
        top = max(8, min(512, 512 * 20 // w))
        ci, co = _log(rng, 3, top), _log(rng, 8, top)
        if rng.random() < 0.6:
            ci, co = max(16, ci // 16 * 16), max(16, co // 16 * 16)
        k = rng.choice((1, 3, 3))
        return _conv(None, ci, co, h, w, k, 1 if k == 1 else rng.choice((1, 1, 2)), batch=rng.choice((1, 1, 1, 2, 4)),
                     x=rng.choice(("f16", "f16", "f32")), out=rng.choice(("f16", "f32")),
                     residual=rng.random() < 0.25, act=rng.choice(("SILU", "SILU", "RELU", "NONE")))
    hkv, d = rng.choice((2, 4, 8)), rng.choice((64, 128))
    hq = hkv * rng.choice((1, 2, 4))
    cache = 256 * rng.randint(1, 16)
    return {"op": "decoder", "layers": rng.randint(2, 6), "dim": 128 * rng.randint(6, 16), "hq": hq, "hkv": hkv, "d": d,
            "ffn": 128 * rng.randint(16, 64), "vocab": 64 * rng.randint(32, 256), "cache": cache,
            "count": rng.randint(1, cache - 1)}


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _size(rng, lo, hi):
    """A layer width: mostly a multiple of 128 or 64, sometimes of 8, sometimes odd."""
    n = _log(rng, lo, hi)
    step = rng.choice((128, 128, 128, 64, 64, 8, 1))
    return max(lo, n // step * step)


def _named(name, case):
    return dict(case, name=name) if name else case


def _linear(name, m, k, n, x="f16", w="f16", out="f32", bias=False, residual=False, act="NONE", gated=False):
    return _named(name, {"op": "linear", "m": m, "k": k, "n": n, "x": x, "w": w, "out": out, "bias": bias,
                         "residual": residual, "act": act, "gated": gated})


def _attention(name, hq, hkv, d, t, x="f16", kv=None, out="f16", causal=True, span=0, cache=0, count=0):
    return _named(name, {"op": "attention", "hq": hq, "hkv": hkv, "d": d, "t": t, "x": x, "kv": kv or x, "out": out,
                         "causal": causal, "span": span, "cache": cache, "count": count})


def _conv(name, ci, co, h, w, k, stride, batch=1, x="f16", out="f32", residual=False, act="SILU"):
    return _named(name, {"op": "conv", "batch": batch, "ci": ci, "co": co, "h": h, "w": w, "k": k, "stride": stride,
                         "x": x, "out": out, "residual": residual, "act": act})


# ---- inputs ------------------------------------------------------------------

class _Dev:
    """A torch tensor as the buffer handle _capi's argument builders take."""

    def __init__(self, t):
        self.t, self.ptr, self.shape = t, t.data_ptr(), tuple(t.shape)
        self.nbytes = t.numel() * t.element_size()
        self.code = {torch.float32: capi.F32, torch.float16: capi.F16}.get(t.dtype)


class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, shape, dtype, sigma=1.0):
        return (torch.randn(shape, generator=self.g, device="cuda") * sigma).to(TORCH[dtype])

    def uniform(self, shape, dtype):
        return (torch.rand(shape, generator=self.g, device="cuda") * 2 - 1).to(TORCH[dtype])


def _inputs(case, seed):
    """The tensors of a case from its seed: what both prepare() and exact() start from."""
    r, c = _Rand(seed), case
    if c["op"] == "linear":
        bdt = c["w"]
        t = {"w": r.normal((c["n"], c["k"]), c["w"], 0.02)}
        if c["bias"]:
            t["bias"] = r.normal((c["n"],), bdt, 0.02)
        t["x"] = r.normal((c["m"], c["k"]), c["x"])
        if c["residual"]:
            t["residual"] = r.normal((c["m"], c["n"]), c["out"])
        return t
    if c["op"] == "attention":
        t = {"q": r.normal((1, c["hq"], c["t"], c["d"]), c["x"]),
             "k": r.normal((1, c["hkv"], c["t"], c["d"]), c["x"]),
             "v": r.normal((1, c["hkv"], c["t"], c["d"]), c["x"])}
        if c["cache"]:
            t["kc"] = r.normal((c["hkv"], c["cache"], c["d"]), c["kv"])
            t["vc"] = r.normal((c["hkv"], c["cache"], c["d"]), c["kv"])
        return t
    if c["op"] == "scores":
        return {"q": r.normal((1, c["hq"], c["tq"], c["d"]), c["x"]),
                "k": r.normal((1, c["hkv"], c["tkv"], c["d"]), c["x"])}
    if c["op"] == "conv":
        t = {"w": r.normal((c["co"], c["ci"], c["k"], c["k"]), "f16", 1.0 / math.sqrt(c["ci"] * c["k"] * c["k"])),
             "bias": r.normal((c["co"],), "f16", 0.02), "x": r.uniform((c["batch"], c["ci"], c["h"], c["w"]), c["x"])}
        if c["residual"]:
            t["residual"] = r.normal((c["batch"], c["co"], _out(c["h"], c), _out(c["w"], c)), c["x"])
        return t
    t = {"x": r.normal((1, c["dim"]), "f16"), "head": r.normal((c["vocab"], c["dim"]), "f16", c["dim"] ** -0.5)}
    for i in range(c["layers"]):
        for name, n, k in (("wqkv", (c["hq"] + 2 * c["hkv"]) * c["d"], c["dim"]), ("wo", c["dim"], c["hq"] * c["d"]),
                           ("wgu", 2 * c["ffn"], c["dim"]), ("wd", c["dim"], c["ffn"])):
            t[f"{name}{i}"] = r.normal((n, k), "f16", 0.7 * k ** -0.5)
        for name in ("kc", "vc"):
            t[f"{name}{i}"] = r.normal((c["hkv"], c["cache"], c["d"]), "f16")
    return t


def _out(n, c):
    return (n - 1) // c["stride"] + 1


def _linear_call(out, x, w, bias=None, residual=None, act="NONE", gated=False):
    """The argument struct of a Linear, with its packed weight and workspace, and what they keep alive."""
    a = capi.linear_args(_Dev(out), _Dev(x), _Dev(w), None if bias is None else _Dev(bias),
                         None if residual is None else _Dev(residual), epi=act, gated=gated, gate_epi="SILU")
    a.bias_repeat = a.N if bias is not None else 0     # one bias row for every output row
    packed = capi.linear_pack_weight(a)
    if packed is not None:
        a.packed_weight = packed.ptr
    ws = _workspace(a, capi.linear_workspace_size(a))
    return a, (packed, ws)


def _workspace(a, need):
    if not need:
        return None
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    a.workspace, a.workspace_bytes = ws.data_ptr(), need
    return ws


def prepare(case, seed):
    c, L = case, capi.lib()
    t = _inputs(c, seed)
    stream = torch.cuda.current_stream().cuda_stream
    if c["op"] == "linear":
        n = c["n"] // 2 if c["gated"] else c["n"]
        out = torch.empty((c["m"], n), dtype=TORCH[c["out"]], device="cuda")
        a, keep = _linear_call(out, t["x"], t["w"], t.get("bias"), t.get("residual"), c["act"], c["gated"])
        return {"call": L.vai_linear_launch, "args": ctypes.byref(a), "stream": stream, "out": out, "keep": (a, keep, t)}
    if c["op"] == "attention":
        out = torch.empty((1, c["t"], c["hq"], c["d"]), dtype=TORCH[c["out"]], device="cuda")
        a, keep = _attention_call(out, t["q"], t["k"], t["v"], c, t.get("kc"), t.get("vc"))
        outs = (out, t["kc"], t["vc"]) if c["cache"] else out
        return {"call": L.vai_attention_launch, "args": ctypes.byref(a), "stream": stream, "out": outs,
                "keep": (a, keep, t)}
    if c["op"] == "scores":
        out = torch.empty((1, c["hq"], c["tq"], c["tkv"]), dtype=torch.float32, device="cuda")
        a = capi.attn_scores_args(_Dev(out), _Dev(t["q"]), _Dev(t["k"]), causal=True, span=c["span"])
        return {"call": L.vai_attn_scores_launch, "args": ctypes.byref(a), "stream": stream, "out": out, "keep": (a, t)}
    if c["op"] == "conv":
        out = torch.empty((c["batch"], c["co"], _out(c["h"], c), _out(c["w"], c)), dtype=TORCH[c["out"]], device="cuda")
        a = capi.conv2d_args(_Dev(out), _Dev(t["x"]), _Dev(t["w"]), _Dev(t["bias"]), None,
                             _Dev(t["residual"]) if c["residual"] else None, stride=c["stride"], epi=c["act"])
        packed = capi.conv2d_pack_weight(a)
        if packed is not None:
            a.packed_weight = packed.ptr
        ws = _workspace(a, capi.conv2d_workspace_size(a))
        return {"call": L.vai_conv2d_launch, "args": ctypes.byref(a), "stream": stream, "out": out,
                "keep": (a, packed, ws, t)}
    return _prepare_decoder(c, t)


def _attention_call(out, q, k, v, c, kc=None, vc=None):
    count = cache = None
    if kc is not None:
        count = torch.tensor([c["count"]], dtype=torch.int32, device="cuda")
        cache = (_Dev(kc), _Dev(vc), _Dev(count), False)
    a = capi.attention_args(_Dev(out), _Dev(q), _Dev(k), _Dev(v), causal=c["causal"], span=c["span"], cache=cache)
    ws = _workspace(a, capi.lib().vai_attention_workspace_size(ctypes.byref(a)))
    return a, (count, ws)


def _prepare_decoder(c, t):
    """One token's step, recorded once: per layer the q/k/v projection, attention over the layer's cache, the
    output projection with its residual, and the gated MLP with its residual; then the head."""
    L, d, hq, hkv = capi.lib(), c["d"], c["hq"], c["hkv"]
    new = lambda n, dt=torch.float16: torch.empty((1, n), dtype=dt, device="cuda")  # noqa: E731
    calls, keep, x = [], [t], t["x"]

    def linear(*args, **kw):
        a, kept = _linear_call(*args, **kw)
        calls.append((L.vai_linear_launch, a))
        keep.append((args, kw, kept))
        return args[0]

    for i in range(c["layers"]):
        qkv = linear(new((hq + 2 * hkv) * d), x, t[f"wqkv{i}"])
        q, k, v = qkv.view(-1, 1, d).split((hq, hkv, hkv))
        att = new(hq * d)
        a, kept = _attention_call(att.view(1, 1, hq, d), q[None], k[None], v[None],
                                  {"causal": True, "span": 0, "count": c["count"]}, t[f"kc{i}"], t[f"vc{i}"])
        calls.append((L.vai_attention_launch, a))
        keep.append((qkv, att, kept))
        x = linear(new(c["dim"]), att, t[f"wo{i}"], None, x)
        hidden = linear(new(c["ffn"]), x, t[f"wgu{i}"], gated=True)
        x = linear(new(c["dim"]), hidden, t[f"wd{i}"], None, x)
    logits = linear(new(c["vocab"], torch.float32), x, t["head"])
    torch.cuda.synchronize()
    stream = capi.Stream()

    def record():
        for fn, a in calls:
            capi.check(fn(ctypes.byref(a), stream.ptr), "record")

    graph = capi.Graph(stream, record)
    caches = [t[f"{n}{i}"] for i in range(c["layers"]) for n in ("kc", "vc")]
    return {"graph": graph, "out": (logits, x, caches), "keep": (calls, keep, stream)}


def run(state):
    if "graph" in state:
        state["graph"].launch()
    else:
        st = state["call"](state["args"], state["stream"])
        if st:
            capi.check(st, "launch")
    return state["out"]


# ---- work, tolerances, 64-bit results -----------------------------------------

def _visible(t, base, causal, span):
    """(query, key) pairs the mask leaves t queries behind base earlier keys, and keys some query sees."""
    pairs, first, last = 0, None, 0
    for i in range(t):
        pos = base + i
        end = pos + 1 if causal else base + t
        beg = max(0, pos + 1 - span) if span else 0
        pairs += max(0, end - beg)
        first = beg if first is None else min(first, beg)
        last = max(last, end)
    return pairs, last - first


def work(case):
    c = case
    if c["op"] == "linear":
        m, k, n = c["m"], c["k"], c["n"]
        no = n // 2 if c["gated"] else n
        bytes_ = n * k * BYTES[c["w"]] + m * k * BYTES[c["x"]] + m * no * BYTES[c["out"]] * (2 if c["residual"] else 1)
        return {"bytes": bytes_ + (n * BYTES[c["w"]] if c["bias"] else 0), "flops": 2 * m * n * k}
    if c["op"] == "attention":
        pairs, keys = _visible(c["t"], c["count"], c["causal"], c["span"])
        new = c["t"] * c["hkv"] * c["d"] * 2
        old = max(0, keys - c["t"]) * c["hkv"] * c["d"] * 2
        bytes_ = c["t"] * c["hq"] * c["d"] * (BYTES[c["x"]] + BYTES[c["out"]]) + new * BYTES[c["x"]] + old * BYTES[c["kv"]]
        return {"bytes": bytes_ + (new * BYTES[c["kv"]] if c["cache"] else 0), "flops": 4 * c["d"] * c["hq"] * pairs}
    if c["op"] == "scores":
        pairs, _ = _visible(c["tq"], c["tkv"] - c["tq"], True, c["span"])
        bytes_ = (c["hq"] * c["tq"] + c["hkv"] * c["tkv"]) * c["d"] * BYTES[c["x"]] + c["hq"] * c["tq"] * c["tkv"] * 4
        return {"bytes": bytes_, "flops": 2 * c["d"] * c["hq"] * pairs}
    if c["op"] == "conv":
        pos, wsz = c["batch"] * _out(c["h"], c) * _out(c["w"], c), c["co"] * c["ci"] * c["k"] * c["k"]
        bytes_ = c["batch"] * c["ci"] * c["h"] * c["w"] * BYTES[c["x"]] + (wsz + c["co"]) * 2 + pos * c["co"] * BYTES[c["out"]]
        return {"bytes": bytes_ + (pos * c["co"] * BYTES[c["x"]] if c["residual"] else 0), "flops": 2 * pos * wsz}
    qkv = (c["hq"] + 2 * c["hkv"]) * c["d"]
    weights = c["layers"] * (c["dim"] * (qkv + c["hq"] * c["d"] + 3 * c["ffn"])) + c["dim"] * c["vocab"]
    cached = c["layers"] * 2 * c["hkv"] * c["d"] * (c["count"] + 1)
    return {"bytes": 2 * (weights + cached + 2 * c["dim"]) + 4 * c["vocab"],
            "flops": 2 * weights + c["layers"] * 4 * c["hq"] * c["d"] * (c["count"] + 1)}


def tolerance(case):
    """About four times the largest error against exact() over the listed cases and eighty drawn ones."""
    c = case
    if c["op"] == "linear":
        if c["x"] == "f32" and c["w"] == "f16" and c["m"] > 8:
            return {"rel": 1.2e-3, "max": 1.2e-2}  # activations enter the matrix cores as fp16
        if c["out"] == "f16":
            return {"rel": 8.5e-4, "max": 2e-3}    # one fp16 rounding of the result
        return {"rel": 2.4e-6, "max": 3e-5}        # fp32 sums in another order
    if c["op"] == "attention":
        return {"rel": 2e-3, "max": 2e-2}          # probabilities (and fp32 Q, K, V) enter as fp16
    if c["op"] == "scores":
        return {"rel": 1e-6, "max": 5e-6}
    if c["op"] == "conv":
        if c["x"] == "f32":
            return {"rel": 1.2e-3, "max": 6e-3}    # the input enters the matrix cores as fp16
        return {"rel": 8.5e-4, "max": 2e-3} if c["out"] == "f16" else {"rel": 1e-6, "max": 5e-6}
    return {"rel": 3.2e-3, "max": 1.3e-2}          # fp16 between some twenty layers


def _act(x, name):
    if name == "SILU":
        return x * torch.sigmoid(x)
    if name == "GELU_TANH":
        return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))
    return torch.relu(x) if name == "RELU" else x


def _exact_linear(x, w, bias=None, residual=None, act="NONE", gated=False):
    y = x.double() @ w.double().t()
    if bias is not None:
        y = y + bias.double()
    if gated:
        g, u = y.chunk(2, -1)
        return _act(g, "SILU") * u
    y = _act(y, act)
    return y if residual is None else y + residual.double()


def _exact_attention(q, k, v, causal, span, base):
    """q [hq, t, d], k / v [hkv, base + t, d] with the t new rows last -> [1, t, hq, d]."""
    hq, t, d = q.shape
    g, n = hq // k.shape[0], k.shape[1]
    pos = torch.arange(t, device=q.device)[:, None] + base
    key = torch.arange(n, device=q.device)[None, :]
    see = key <= pos if causal else torch.ones((t, n), dtype=torch.bool, device=q.device)
    if span:
        see = see & (key > pos - span)
    out = torch.empty((1, t, hq, d), dtype=torch.float64, device=q.device)
    for h in range(hq):
        s = q[h].double() @ k[h // g].double().t() / math.sqrt(d)
        out[0, :, h] = torch.softmax(s.masked_fill(~see, -math.inf), -1) @ v[h // g].double()
    return out


def exact(case, seed):
    c, t = case, _inputs(case, seed)
    if c["op"] == "linear":
        return _exact_linear(t["x"], t["w"], t.get("bias"), t.get("residual"), c["act"], c["gated"])
    if c["op"] == "attention":
        if not c["cache"]:
            return _exact_attention(t["q"][0], t["k"][0], t["v"][0], c["causal"], c["span"], 0)
        kc, vc = _appended(t["kc"], t["k"], c["count"]), _appended(t["vc"], t["v"], c["count"])
        n = c["count"] + c["t"]
        return _exact_attention(t["q"][0], kc[:, :n], vc[:, :n], c["causal"], c["span"], c["count"]), kc, vc
    if c["op"] == "scores":
        g, off = c["hq"] // c["hkv"], c["tkv"] - c["tq"]
        pos = torch.arange(c["tq"], device="cuda")[:, None] + off
        key = torch.arange(c["tkv"], device="cuda")[None, :]
        hide = key > pos
        if c["span"]:
            hide = hide | (key < pos + 1 - c["span"])
        k = t["k"].double().repeat_interleave(g, 1)
        return (t["q"].double() @ k.transpose(-1, -2) / math.sqrt(c["d"])).masked_fill(hide, -math.inf)
    if c["op"] == "conv":
        w = t["w"].double().reshape(c["co"], -1)
        outs = []
        for x in t["x"]:      # an image at a time: the unfolded input is k*k times its size
            cols = torch.nn.functional.unfold(x.double()[None], c["k"], padding=c["k"] // 2, stride=c["stride"])[0]
            outs.append((w @ cols).view(c["co"], _out(c["h"], c), _out(c["w"], c)))
        y = _act(torch.stack(outs) + t["bias"].double()[:, None, None], c["act"])
        return y + t["residual"].double() if c["residual"] else y
    x, caches = t["x"].double(), []
    for i in range(c["layers"]):
        qkv = _exact_linear(x, t[f"wqkv{i}"])
        q, k, v = qkv.view(-1, 1, c["d"]).split((c["hq"], c["hkv"], c["hkv"]))
        kc, vc = (_appended(t[f"{n}{i}"].double(), y[None], c["count"]) for n, y in (("kc", k), ("vc", v)))
        caches += [kc, vc]
        n = c["count"] + 1
        att = _exact_attention(q, kc[:, :n], vc[:, :n], True, 0, c["count"])
        x = _exact_linear(att.view(1, -1), t[f"wo{i}"], None, x)
        x = _exact_linear(_exact_linear(x, t[f"wgu{i}"], gated=True), t[f"wd{i}"], None, x)
    return _exact_linear(x, t["head"]), x, caches


def _appended(cache, new, count):
    c = cache.double().clone()
    c[:, count:count + new.shape[2]] = new[0].double()
    return c
