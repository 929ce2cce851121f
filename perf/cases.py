"""What a program that serves or loads a W4A16 model has this library do, as cases that can be timed.

Every case goes through the public entry points: the Python mirror of the reference's interface (tensorwarp_amd) and,
where the mirror has no function that takes the caller's own buffers, the C ABI of include/twmarlin.h itself.  Arrays are
torch tensors handed over by pointer, as include/twmarlin.h describes; work runs on the context's own stream.

kind        a pass is
decode      one decode step's linear layers of `layers` transformer layers for `m` sequences, replayed as one captured
            graph: fused QKV with the split (and the biases) in the store, the output projection, gate+up with the SwiGLU
            gate in the store, and the down projection on that call's f32 rows
prefill     the same calls for `m` prompt tokens, issued one by one: the row count changes from prompt to prompt, so
            nothing is captured
reference   the drop-in entry point on the reference's own arrays, f32 rows, one row: the four projections of each layer
            issued one by one
lm_head     logits of `m` rows over the vocabulary and the greedy token of each, as one graph
moe         the expert part of `layers` mixture-of-experts layers for one token: the routed gate+up projections with the
            GEGLU gate in the store, then the weighted down projections added to the residual row; one graph
format      loading an unquantized gate and up matrix: quantize both from f32, fuse them along N, and unpack the result to
            the f16 matrix that the FP16 route multiplies with
"""
import math

import torch

import tensorwarp_amd as T
from tensorwarp_amd import _lib

_NAMES = {torch.float32: "f32", torch.float16: "f16", torch.uint8: "u8", torch.int32: "i32"}


def listed():
    qwen05 = {"hidden": 896, "kv": 128, "ffn": 4864, "bias": True}
    qwen7 = {"hidden": 3584, "kv": 512, "ffn": 18944, "bias": True}
    llama7 = {"hidden": 4096, "kv": 4096, "ffn": 11008, "bias": False}
    return [
        # the small model's whole decode step, one user: 96 launches of 2 - 3 us each
        dict({"name": "decode_qwen05b_m1", "kind": "decode", "m": 1, "layers": 24, "rows": "f16"}, **qwen05),
        # single-user decode of the 7B model, the reference's headline workload
        dict({"name": "decode_qwen7b_m1", "kind": "decode", "m": 1, "layers": 4, "rows": "f16"}, **qwen7),
        # a few users at once
        dict({"name": "decode_qwen7b_m8", "kind": "decode", "m": 8, "layers": 4, "rows": "f16"}, **qwen7),
        # a full decode batch
        dict({"name": "decode_qwen7b_m32", "kind": "decode", "m": 32, "layers": 4, "rows": "f16"}, **qwen7),
        # an odd batch of f32 rows (the reference's decode buffers are f32)
        dict({"name": "decode_llama7b_m13_f32", "kind": "decode", "m": 13, "layers": 4, "rows": "f32"}, **llama7),
        # a program that keeps the reference's arrays and changes only the call
        dict({"name": "reference_qwen7b_m1", "kind": "reference", "layers": 2}, **qwen7),
        # the vocabulary projection of a greedy decode step
        {"name": "lm_head_qwen7b_m1", "kind": "lm_head", "m": 1, "hidden": 3584, "vocab": 152064, "rows": "f16"},
        # mixture-of-experts decode, eight of 128 experts
        {"name": "moe_128x704_top8", "kind": "moe", "hidden": 2816, "dim": 704, "experts": 128, "top_k": 8, "layers": 2},
        # a short prompt, or a decode batch beyond 32 rows
        dict({"name": "prefill_qwen7b_m96", "kind": "prefill", "m": 96, "layers": 2, "rows": "f16"}, **qwen7),
        # an ordinary prompt and a long one
        dict({"name": "prefill_llama7b_m512", "kind": "prefill", "m": 512, "layers": 1, "rows": "f16"}, **llama7),
        dict({"name": "prefill_llama7b_m2048", "kind": "prefill", "m": 2048, "layers": 1, "rows": "f16"}, **llama7),
        # model load
        {"name": "format_3584x18944", "kind": "format", "k": 3584, "n": 18944, "nk": True},
    ]


def _log_int(rng, lo, hi, step=1):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "reference", "lm_head", "moe", "format"])
    if kind == "lm_head":
        return {"kind": kind, "m": _log_int(rng, 1, 16), "hidden": _log_int(rng, 896, 4096, 64),
                "vocab": _log_int(rng, 32000, 152064), "rows": rng.choice(["f16", "f32"])}
    if kind == "moe":
        return {"kind": kind, "hidden": _log_int(rng, 1024, 4096, 64), "dim": _log_int(rng, 384, 1536, 32),
                "experts": rng.choice([8, 16, 32, 64, 128]), "top_k": rng.choice([1, 2, 4, 6, 8]), "layers": 2}
    if kind == "format":
        return {"kind": kind, "k": _log_int(rng, 896, 4096, 32), "n": _log_int(rng, 1024, 18944), "nk": rng.random() < 0.5}
    hidden = _log_int(rng, 896, 4096, 64 if rng.random() < 0.8 else 32)
    kv = min(hidden, 64 * rng.choice([2, 4, 8, 16])) if rng.random() < 0.8 else hidden
    ffn = min(18944, int(hidden * rng.uniform(2.5, 5.5)) // 32 * 32)
    case = {"kind": kind, "hidden": hidden, "kv": kv, "ffn": ffn, "bias": rng.random() < 0.5, "layers": 2 if kind != "prefill" else 1}
    if kind == "decode":
        # below about 250 MB a pass would be served from the cache that a whole model does not fit
        layer = (hidden * (2 * hidden + 2 * kv + 3 * ffn)) * 9 // 16
        case["layers"] = max(2, min(24, 120_000_000 // layer))
        case["m"], case["rows"] = _log_int(rng, 1, 32), rng.choice(["f16", "f16", "f32"])
    elif kind == "prefill":
        # a drawn layer has up to 1.5 times the weights of the longest listed prompt's, so its prompts end earlier
        case["m"], case["rows"] = _log_int(rng, 33, 1280), rng.choice(["f16", "f16", "f32"])
    return case


class _Rows:
    """A torch tensor as the mirror's functions take their arguments: a pointer and the name of the element type."""

    def __init__(self, t):
        self.tensor, self.ptr, self.dtype, self.numel = t, t.data_ptr(), _NAMES[t.dtype], t.numel()


class _State:
    """What a program holds between calls; frees the library's objects with it."""

    def __init__(self, case):
        self.case, self.owned, self.kept, self.graph = dict(case), [], [], None

    def rows(self, t):
        v = _Rows(t)
        self.kept.append(v)
        return v

    def own(self, handle):
        self.owned.append(handle)
        return handle

    def __del__(self):
        if self.graph is not None:
            self.graph.destroy()
        for h in self.owned:
            h.free()


_device = None


def _dev():
    """The process's one context."""
    global _device
    if _device is None:
        _device = T.WarpDevice(0)
    return _device


def _nibbles(gen, g, n):
    """A TW-Marlin pair as a quantized matrix of normally distributed weights has it: nibbles around 8, positive scales."""
    def half():
        return torch.randn(g, n, 16, device="cuda", generator=gen).mul_(2.7).add_(8.5).clamp_(0.0, 15.5).to(torch.uint8)
    packed = half() | (half() << 4)
    scales = (0.006 * (1.0 + 0.25 * torch.randn(g, n, device="cuda", generator=gen)).clamp_(0.3, 2.0)).to(torch.float16)
    return packed, scales


def _activations(gen, m, k, dtype):
    """Normalized rows: order one, with the few large channels that trained models have."""
    a = torch.randn(m, k, device="cuda", generator=gen)
    a[:, torch.randint(0, k, (max(1, k // 256),), device="cuda", generator=gen)] *= 12.0
    return a.to(torch.float32 if dtype == "f32" else torch.float16)


def _weight(s, gen, k, n):
    p, c = _nibbles(gen, k // 32, n)
    torch.cuda.synchronize()
    w = s.own(T.MarlinWeight.from_device(_dev(), _Rows(p), _Rows(c), k, n))
    _dev().synchronize()
    return w


def _out(s, *shape):
    t = torch.zeros(*shape, device="cuda")
    return t, [s.rows(t[i]) for i in range(shape[0])]


def _prepare_layers(s, gen):
    c = s.case
    h, kv, ffn, m, layers = c["hidden"], c["kv"], c["ffn"], c["m"], c["layers"]
    s.layers = []
    for _ in range(layers):
        w = {"qkv": _weight(s, gen, h, h + 2 * kv), "o": _weight(s, gen, h, h)}
        gate, up = _nibbles(gen, h // 32, ffn), _nibbles(gen, h // 32, ffn)
        torch.cuda.synchronize()
        w["gate_up"] = s.own(T.MarlinWeight.gate_up(_dev(), tuple(map(_Rows, gate)), tuple(map(_Rows, up)), h, ffn))
        _dev().synchronize()
        del gate, up
        w["down"] = _weight(s, gen, ffn, h)
        w["biases"] = [s.rows(0.1 * torch.randn(n, device="cuda", generator=gen)) for n in (h, kv, kv)] if c["bias"] else None
        # the rows that the norms and the attention between the projections leave
        w["x"], w["attn"], w["y"] = (s.rows(_activations(gen, m, h, c["rows"])) for _ in range(3))
        s.layers.append(w)
    s.outs = {}
    for name, n in (("q", h), ("k", kv), ("v", kv), ("o", h), ("act", ffn), ("down", h)):
        s.outs[name], views = _out(s, layers, m, n)
        for w, v in zip(s.layers, views):
            w["out_" + name] = v


def _run_layers(s):
    c, dev = s.case, _dev()
    m, ns = c["m"], [c["hidden"], c["kv"], c["kv"]]
    for w in s.layers:
        T.gemm_split(dev, w["qkv"], w["x"], m, [w["out_q"], w["out_k"], w["out_v"]], ns, biases=w["biases"])
        T.gemm(dev, w["o"], w["attn"], m, w["out_o"])
        T.gemm_swiglu(dev, w["gate_up"], w["y"], m, w["out_act"])
        T.gemm(dev, w["down"], w["out_act"], m, w["out_down"])
    return s.outs


def _prepare_reference(s, gen):
    c = s.case
    s.calls, s.outs = [], {}
    shapes = {"qkv": (c["hidden"], c["hidden"] + 2 * c["kv"]), "o": (c["hidden"], c["hidden"]),
              "gate_up": (c["hidden"], 2 * c["ffn"]), "down": (c["ffn"], c["hidden"])}
    views = {}
    for name, (k, n) in shapes.items():
        s.outs[name], views[name] = _out(s, c["layers"], 1, n)
    for i in range(c["layers"]):
        for name, (k, n) in shapes.items():
            p, sc = _nibbles(gen, k // 32, n)
            s.calls.append((s.rows(_activations(gen, 1, k, "f32")), s.rows(p), s.rows(sc), views[name][i], n, k))


def _run_reference(s):
    dev = _dev()
    for call in s.calls:
        T.gemm_tw_marlin_m1(dev, *call)
    return s.outs


def _prepare_lm_head(s, gen):
    c = s.case
    s.w = _weight(s, gen, c["hidden"], c["vocab"])
    s.x = s.rows(_activations(gen, c["m"], c["hidden"], c["rows"]))
    logits = torch.zeros(c["m"], c["vocab"], device="cuda")
    tokens = torch.zeros(c["m"], dtype=torch.int32, device="cuda")
    s.logits, s.tokens = s.rows(logits), s.rows(tokens)
    s.outs = {"logits": logits, "tokens": tokens}


def _run_lm_head(s):
    c = s.case
    T.gemm(_dev(), s.w, s.x, c["m"], s.logits)
    T.argmax(_dev(), s.logits, s.tokens, c["m"], c["vocab"])
    return s.outs


def _bank(s, gen, k, n, experts, paired):
    parts = [_nibbles(gen, k // 32, n) for _ in range(experts)]
    packed, scales = torch.stack([p for p, _ in parts]), torch.stack([c for _, c in parts])
    torch.cuda.synchronize()
    b = s.own(T.ExpertBank.from_device(_dev(), _Rows(packed), _Rows(scales), k // 32 * n * 16, k // 32 * n, k, n, experts, paired))
    _dev().synchronize()
    return b


def _prepare_moe(s, gen):
    c = s.case
    h, dim, top = c["hidden"], c["dim"], c["top_k"]
    acc, accs = _out(s, c["layers"], 1, h)
    gated, gateds = _out(s, c["layers"], top, dim)
    s.outs, s.layers = {"acc": acc, "gated": gated}, []
    for i in range(c["layers"]):
        ids = torch.randperm(c["experts"], device="cuda", generator=gen)[:top].to(torch.float32)
        weights = torch.softmax(torch.randn(top, device="cuda", generator=gen), 0)
        s.layers.append({"gate_up": _bank(s, gen, h, 2 * dim, c["experts"], True), "down": _bank(s, gen, dim, h, c["experts"], False),
                         "x": s.rows(_activations(gen, 1, h, "f32")), "residual": s.rows(torch.randn(1, h, device="cuda", generator=gen)),
                         "ids": s.rows(ids), "weights": s.rows(weights), "gated": gateds[i], "acc": accs[i]})


def _run_moe(s):
    c, dev = s.case, _dev()
    for w in s.layers:
        T.quantize._check(_lib.load().twm_memcpy_d2d(dev.handle, w["acc"].ptr, w["residual"].ptr, 4 * c["hidden"]))
        T.batched_marlin_gate_up(dev, w["x"], w["gate_up"], w["ids"], w["gated"], c["top_k"], act=T.ACT_GEGLU)
        T.batched_marlin_down_axpy(dev, w["gated"], w["down"], w["ids"], w["weights"], w["acc"], c["top_k"])
    return s.outs


def _prepare_format(s, gen):
    k, n = s.case["k"], s.case["n"]
    shape = (n, k) if s.case["nk"] else (k, n)
    s.w = [s.rows(0.02 * torch.randn(*shape, device="cuda", generator=gen)) for _ in range(2)]
    g = k // 32
    s.parts = [(s.rows(torch.zeros(g, n, 16, dtype=torch.uint8, device="cuda")),
                s.rows(torch.zeros(g, n, dtype=torch.float16, device="cuda"))) for _ in range(2)]
    packed = torch.zeros(g, 2 * n, 16, dtype=torch.uint8, device="cuda")
    scales = torch.zeros(g, 2 * n, dtype=torch.float16, device="cuda")
    dense = torch.zeros(k, 2 * n, dtype=torch.float16, device="cuda")
    s.packed, s.scales, s.dense = s.rows(packed), s.rows(scales), s.rows(dense)
    s.outs = {"packed": packed, "scales": scales, "dense": dense}


def _run_format(s):
    import ctypes
    lib, check, h = _lib.load(), T.quantize._check, _dev().handle
    k, n = s.case["k"], s.case["n"]
    for w, (p, c) in zip(s.w, s.parts):
        check(lib.twm_quantize_f32_to_tw_marlin(h, w.ptr, int(s.case["nk"]), k, n, p.ptr, c.ptr))
    ps, cs = ((ctypes.c_void_p * 2)(*[part[i].ptr for part in s.parts]) for i in (0, 1))
    check(lib.twm_fuse_tw_marlin_n(h, ps, cs, k, (ctypes.c_uint32 * 2)(n, n), 2, s.packed.ptr, s.scales.ptr))
    check(lib.twm_dequant_to_f16(h, s.packed.ptr, s.scales.ptr, k, 2 * n, s.dense.ptr))
    return s.outs


_KINDS = {"decode": (_prepare_layers, _run_layers), "prefill": (_prepare_layers, _run_layers),
          "reference": (_prepare_reference, _run_reference), "lm_head": (_prepare_lm_head, _run_lm_head),
          "moe": (_prepare_moe, _run_moe), "format": (_prepare_format, _run_format)}
_CAPTURED = ("decode", "lm_head", "moe")


def prepare(case, seed):
    s = _State(case)
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    _KINDS[case["kind"]][0](s, gen)
    torch.cuda.synchronize()
    if case["kind"] in _CAPTURED:
        s.graph = T.GraphCapture.record_with_device(_dev(), lambda: _KINDS[case["kind"]][1](s))
    return s


def run(state):
    if state.graph is not None:
        state.graph.replay()
        return state.outs
    return _KINDS[state.case["kind"]][1](state)


def _linear(m, k, n, row_bytes, n_out=None):
    return {"bytes": k * n // 2 + k // 32 * n * 2 + m * k * row_bytes + m * (n if n_out is None else n_out) * 4, "flops": 2 * m * k * n}


def work(case):
    c = case
    if c["kind"] == "format":
        kn = c["k"] * c["n"]
        # f32 in, the fused 4.5-bit arrays and the f16 matrix out, for two matrices
        return {"bytes": 2 * (4 * kn + kn // 2 + kn // 16 + 2 * kn), "flops": 0}
    es = 2 if c.get("rows") == "f16" else 4
    if c["kind"] == "lm_head":
        parts = [_linear(c["m"], c["hidden"], c["vocab"], es)]
    elif c["kind"] == "moe":
        top, h, dim = c["top_k"], c["hidden"], c["dim"]
        one = [_linear(1, h, 2 * dim, 0, dim), _linear(1, dim, h, 0, 0)]
        parts = one * top + [{"bytes": 4 * h * 3, "flops": 0}]
    else:
        h, kv, ffn, m = c["hidden"], c["kv"], c["ffn"], c.get("m", 1)
        parts = [_linear(m, h, h + 2 * kv, es), _linear(m, h, h, es),
                 _linear(m, h, 2 * ffn, es, 2 * ffn if c["kind"] == "reference" else ffn), _linear(m, ffn, h, 4)]
    layers = c.get("layers", 1)
    return {k: layers * sum(p[k] for p in parts) for k in ("bytes", "flops")}


def tolerance(case):
    if case["kind"] == "format":
        return "exact"
    if case["kind"] == "prefill":
        # weights and f32 rows are rounded to f16, sums are f32: against the f64 product on the exact weights and rows the
        # outputs are off by 1.7e-4 (qkv, o) to 3.7e-4 (down), 4e-3 at most for a gated value
        return {"rel": 1e-3, "max": 1e-2}
    # exact weights, rows exact (f16) or in two f16 terms, f32 sums: against the f64 product the outputs are off by 7e-8 to
    # 3.3e-7 and single values by up to 3.3e-6, most on the gated products of 32 rows
    return {"rel": 1.5e-6, "max": 1.5e-5}
