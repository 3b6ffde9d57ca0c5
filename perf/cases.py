"""The work a user of the library has it do, as cases that can be timed.

A model's weights live on the device as GGUF blocks.  A decoder multiplies one token's activations with them (``decode``,
``linear`` with m = 1), a server multiplies a few tokens of several sequences (``linear`` with m = 2 ... 300), a prompt is
several hundred to a few thousand tokens (``linear`` and ``prefill``).  A converter turns f32 tensors into blocks and back, on
the device (``quantize``, ``dequantize``) or from and to host memory (``host_codec``).

A model's layers follow one another and each has weights of its own, so a ``linear`` case walks a stack of ``layers`` equal
weights: small batches then read their weights from memory and not from a cache that a single weight would stay in.

``run`` goes through ``GgufLinear.forward``, the batch entry points of the C ABI and ``quantize`` / ``dequantize``.
"""
from __future__ import annotations

import math

import numpy as np
import torch  # before the library is loaded: both then share one HIP runtime

import pmetal_amd as pm
from pmetal_amd import _lib

TYPES = {"q8_0": 8, "q2_k": 10, "q3_k": 11, "q4_k": 12, "q5_k": 13, "q6_k": 14}
BLOCK = {"q8_0": (32, 34), "q2_k": (256, 84), "q3_k": (256, 110), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210)}
NAMES = {v: k for k, v in TYPES.items()}


def listed():
    return [
        # the smallest call: one token through MLP projections of a small model, f32 activations
        {"name": "gemv_q8_0_small", "kind": "linear", "type": "q8_0", "n": 3072, "k": 1024, "m": 1, "layers": 4, "x": "f32", "y": "f32", "order": 0},
        # every projection of one token of a 0.6B-class Q4_K_M model, recorded once and replayed as a decoder submits its step
        {"name": "decode_hidden1024", "kind": "decode", "hidden": 1024, "q": 2048, "kv": 1024, "ffn": 3072, "layers": 28, "vocab": 151936, "replay": True},
        # eight layers of an 8B-class Q4_K_M model, one token, launched one dependent group after the other
        {"name": "decode_hidden4096", "kind": "decode", "hidden": 4096, "q": 4096, "kv": 1024, "ffn": 14336, "layers": 8, "vocab": 0, "replay": False},
        # a decode step of sixteen sequences
        {"name": "linear_q4_k_m16", "kind": "linear", "type": "q4_k", "n": 14336, "k": 4096, "m": 16, "layers": 8, "x": "bf16", "y": "bf16", "order": 0},
        # an odd number of sequences through the down projection, long rows, f32 results
        {"name": "linear_q6_k_m27", "kind": "linear", "type": "q6_k", "n": 4096, "k": 14336, "m": 27, "layers": 6, "x": "bf16", "y": "f32", "order": 0},
        # gate and up projections of 64 tokens: two weights, one activation
        {"name": "pair_q4_k_m64", "kind": "pair", "type": "q4_k", "n": 14336, "k": 4096, "m": 64, "layers": 4, "x": "bf16", "y": "bf16", "order": 0},
        # ragged everything: a short prompt, row count off every tile, f32 activations
        {"name": "linear_q8_0_m203", "kind": "linear", "type": "q8_0", "n": 4999, "k": 3584, "m": 203, "layers": 4, "x": "f32", "y": "f32", "order": 0},
        # a prompt of 512 tokens through one wide projection
        {"name": "linear_q4_k_m512", "kind": "linear", "type": "q4_k", "n": 14336, "k": 4096, "m": 512, "layers": 2, "x": "bf16", "y": "bf16", "order": 0},
        # a prompt of 2048 tokens through all projections of a layer (Q4_K and Q6_K)
        {"name": "prefill_hidden4096_m2048", "kind": "prefill", "hidden": 4096, "q": 4096, "kv": 1024, "ffn": 14336, "m": 2048},
        # converting a model that is on the device: four layers of the 8B-class shape, f32 -> Q4_K_M
        {"name": "quantize_hidden4096", "kind": "quantize", "hidden": 4096, "q": 4096, "kv": 1024, "ffn": 14336, "layers": 4},
        # blocks -> f32 on the device
        {"name": "dequantize_q6_k", "kind": "dequantize", "type": "q6_k", "n": 14336, "k": 4096, "order": 0},
        # the drop-in quantize() / dequantize() on host memory, one MLP tensor of a small model
        {"name": "host_codec_q8_0", "kind": "host_codec", "type": "q8_0", "n": 3072, "k": 1024},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "pair", "decode", "prefill", "quantize", "dequantize", "host_codec"])
    t = rng.choice(["q4_k", "q4_k", "q6_k", "q8_0", "q5_k", "q3_k", "q2_k"])
    if kind in ("linear", "pair"):
        k = 256 * _log_int(rng, 4, 56)
        n = _log_int(rng, 1000, 15000)
        m = rng.choice([1, _log_int(rng, 2, 32), _log_int(rng, 2, 32), _log_int(rng, 33, 300), _log_int(rng, 33, 300), _log_int(rng, 301, 2048)])
        if kind == "pair":
            m = max(m, 2)
        layers = 2 if m > 300 else 4 if n * k > 20_000_000 else 8
        m = min(m, 150_000_000_000 // (n * k * layers * (2 if kind == "pair" else 1)))  # a third of the largest listed case's products
        return {"kind": kind, "type": t, "n": n, "k": k, "m": m, "layers": layers, "x": rng.choice(["bf16", "bf16", "f32"]),
                "y": "f32" if m == 1 else rng.choice(["bf16", "f32"]), "order": rng.choice([0, 1])}
    hidden = 256 * _log_int(rng, 4, 20)
    kv = rng.choice([hidden // 4, hidden // 2, hidden])
    ffn = 256 * round(hidden * rng.uniform(2.5, 3.6) / 256)
    if kind == "decode":
        return {"kind": kind, "hidden": hidden, "q": rng.choice([hidden, hidden + 1024]), "kv": kv, "ffn": ffn, "layers": rng.randint(4, 8),
                "vocab": rng.choice([0, _log_int(rng, 30000, 130000)]), "replay": rng.choice([True, False])}
    if kind == "prefill":
        return {"kind": kind, "hidden": min(hidden, 4096), "q": min(hidden, 4096), "kv": min(kv, 1024), "ffn": min(ffn, 14336), "m": _log_int(rng, 100, 2000)}
    if kind == "quantize":
        return {"kind": kind, "hidden": min(hidden, 4096), "q": min(hidden, 4096), "kv": min(kv, 1024), "ffn": min(ffn, 14336), "layers": rng.randint(1, 4)}
    n, k = _log_int(rng, 500, 14336), 256 * _log_int(rng, 4, 16)
    if kind == "dequantize":
        return {"kind": kind, "type": t, "n": n, "k": k, "order": rng.choice([0, 1])}
    return {"kind": kind, "type": t, "n": _log_int(rng, 100, 3_200_000 // k), "k": k}


# ---- inputs ----
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _stream():
    return torch.cuda.current_stream().cuda_stream or None


def _nbytes(t, elements):
    block, size = BLOCK[t]
    return -(-elements // block) * size


def _weight_values(g, n, k):
    """Trained weights as a quantizer meets them: N(0, 0.02) with one in a thousand at +-0.5."""
    w = torch.randn(n * k, generator=g, device="cuda").mul_(0.02)
    chance = torch.rand(n * k, generator=g, device="cuda")
    return w.masked_fill_(chance < 5e-4, 0.5).masked_fill_(chance > 1 - 5e-4, -0.5)


def _weight(g, t, n, k):
    w = _weight_values(g, n, k)
    blocks = torch.empty(_nbytes(t, n * k), dtype=torch.uint8, device="cuda")
    pm.check(_lib.load().pmetal_hip_quantize_dev(TYPES[t], w.data_ptr(), n * k, blocks.data_ptr(), blocks.numel(), _stream()), "quantize")
    torch.cuda.current_stream().synchronize()  # w goes back to torch's allocator here
    return blocks


def _activations(g, m, k, dtype):
    """N(0, 1) with a few channels far larger than the rest, as the residual stream of a trained model has them."""
    x = torch.randn(m, k, generator=g, device="cuda")
    x[:, torch.randint(0, k, (max(k // 1000, 1),), generator=g, device="cuda")] *= 20.0
    return x.to(torch.bfloat16) if dtype == "bf16" else x


def _dtype(name):
    return pm.DTYPE_BF16 if name == "bf16" else pm.DTYPE_F32


def _torch_dtype(name):
    return torch.bfloat16 if name == "bf16" else torch.float32


def _layer_tensors(c, layers):
    """(GGUF name, rows, columns) of the projections of each layer, in the order a forward pass uses them."""
    h, q, kv, f = c["hidden"], c["q"], c["kv"], c["ffn"]
    return [[(f"blk.{i}.attn_q.weight", q, h), (f"blk.{i}.attn_k.weight", kv, h), (f"blk.{i}.attn_v.weight", kv, h), (f"blk.{i}.attn_output.weight", h, q),
             (f"blk.{i}.ffn_gate.weight", f, h), (f"blk.{i}.ffn_up.weight", f, h), (f"blk.{i}.ffn_down.weight", h, f)] for i in range(layers)]


def _recipe(name, layers):
    return NAMES[int(pm.q4km_tensor_type(name, 2, layers))]


GROUPS = ((0, 1, 2), (3,), (4, 5), (6,))  # q k v | output | gate up | down: what shares an input and waits for nothing in between


def _linear_desc(t, n, k, w, x, y):
    return _lib.LinearDesc(TYPES[t], pm.DTYPE_BF16, 0, 0, n, k, w.data_ptr(), x.data_ptr(), y.data_ptr())


def _prepare_decode(c, g):
    """One list of descriptors per group of projections that a decoder can issue together."""
    lib, keep, calls, filled = _lib.load(), [], [], 0
    widths = [n for tensors in _layer_tensors(c, c["layers"]) for _, n, _ in tensors] + ([c["vocab"]] if c["vocab"] else [])
    out = torch.zeros(sum(-(-n // 16) * 16 for n in widths), device="cuda")  # every projection's results, one behind the other

    def results(n):
        nonlocal filled
        y = out[filled:filled + n]
        filled += -(-n // 16) * 16
        return y

    xs = {name: _activations(g, 1, width, "bf16") for name, width in (("attn", c["hidden"]), ("out", c["q"]), ("ffn", c["hidden"]), ("down", c["ffn"]))}
    for tensors in _layer_tensors(c, c["layers"]):
        for group, xname in zip(GROUPS, ("attn", "out", "ffn", "down")):
            descs = (_lib.LinearDesc * len(group))()
            for i, at in enumerate(group):
                name, n, k = tensors[at]
                t = _recipe(name, c["layers"])
                w = _weight(g, t, n, k)
                descs[i] = _linear_desc(t, n, k, w, xs[xname], results(n))
                keep.append(w)
            calls.append((descs, len(group)))
    if c["vocab"]:
        t = _recipe("output.weight", c["layers"])
        w = _weight(g, t, c["vocab"], c["hidden"])
        descs = (_lib.LinearDesc * 1)(_linear_desc(t, c["vocab"], c["hidden"], w, xs["attn"], results(c["vocab"])))
        keep.append(w), calls.append((descs, 1))
    state = {"kind": "decode", "lib": lib, "calls": calls, "keep": (keep, xs), "out": out, "recording": None}
    if c["replay"]:
        state["recording"] = _Recording(lib, calls)
    return state


class _Recording:
    """A decode step recorded on a stream of its own; destroyed with the state."""

    def __init__(self, lib, calls):
        self.lib, self.stream = lib, lib.pmetal_hip_stream_create()
        torch.cuda.synchronize()
        pm.check(lib.pmetal_hip_record_begin(self.stream))
        for descs, count in calls:
            pm.check(lib.pmetal_hip_qgemv_batch(descs, count, self.stream))
        self.handle = lib.pmetal_hip_record_end(self.stream)
        if not self.handle:
            raise RuntimeError(lib.pmetal_hip_last_error_message())

    def __del__(self):
        torch.cuda.synchronize()
        self.lib.pmetal_hip_recording_destroy(self.handle)
        self.lib.pmetal_hip_stream_destroy(self.stream)


def _gemm_desc(t, n, w, y, y_dtype, order):
    return _lib.GemmDesc(TYPES[t], y_dtype, order, 0, n, w.data_ptr(), y.data_ptr())


def prepare(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    pm.init(torch.cuda.current_device())
    if kind == "linear":
        t, n, k, m = c["type"], c["n"], c["k"], c["m"]
        x = _activations(g, m, k, c["x"])
        stack = [(pm.GgufLinear(TYPES[t], n, k, _weight(g, t, n, k), order=c["order"]), torch.empty(m, n, dtype=_torch_dtype(c["y"]), device="cuda"))
                 for _ in range(c["layers"])]
        return {"kind": kind, "x": x, "m": m, "xd": _dtype(c["x"]), "yd": _dtype(c["y"]), "stack": stack}
    if kind == "pair":
        t, n, k, m, yd = c["type"], c["n"], c["k"], c["m"], _dtype(c["y"])
        x = _activations(g, m, k, c["x"])
        keep, calls = [], []
        for _ in range(c["layers"]):
            ws = [_weight(g, t, n, k) for _ in range(2)]
            ys = [torch.empty(m, n, dtype=_torch_dtype(c["y"]), device="cuda") for _ in range(2)]
            calls.append(((_lib.GemmDesc * 2)(*[_gemm_desc(t, n, w, y, yd, c["order"]) for w, y in zip(ws, ys)]), 2, k, x))
            keep.append((ws, ys))
        return {"kind": "gemm_batches", "lib": _lib.load(), "m": m, "xd": _dtype(c["x"]), "calls": calls, "keep": keep, "outs": [y for _, ys in keep for y in ys]}
    if kind == "decode":
        return _prepare_decode(c, g)
    if kind == "prefill":
        m, keep, calls, outs = c["m"], [], [], []
        tensors = _layer_tensors(c, 1)[0]
        for group in GROUPS:
            k = tensors[group[0]][2]
            x = _activations(g, m, k, "bf16")
            descs = (_lib.GemmDesc * len(group))()
            for i, at in enumerate(group):
                name, n, _ = tensors[at]
                t = _recipe(name, 1)
                w, y = _weight(g, t, n, k), torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
                descs[i] = _gemm_desc(t, n, w, y, pm.DTYPE_BF16, 0)
                keep.append(w), outs.append(y)
            calls.append((descs, len(group), k, x))
        return {"kind": "gemm_batches", "lib": _lib.load(), "m": m, "xd": pm.DTYPE_BF16, "calls": calls, "keep": keep, "outs": outs}
    if kind == "quantize":
        tensors = [(_recipe(name, c["layers"]), n, k) for layer in _layer_tensors(c, c["layers"]) for name, n, k in layer]
        src = [_weight_values(g, n, k) for _, n, k in tensors]
        dst = [torch.empty(_nbytes(t, n * k), dtype=torch.uint8, device="cuda") for t, n, k in tensors]
        descs = (_lib.QuantizeDesc * len(tensors))(*[_lib.QuantizeDesc(TYPES[t], 0, s.data_ptr(), s.numel(), d.data_ptr(), d.numel())
                                                     for (t, _, _), s, d in zip(tensors, src, dst)])
        return {"kind": kind, "lib": _lib.load(), "descs": descs, "src": src, "outs": dst}
    if kind == "dequantize":
        t, n, k = c["type"], c["n"], c["k"]
        return {"kind": kind, "lib": _lib.load(), "t": TYPES[t], "order": c["order"], "blocks": _weight(g, t, n, k), "out": torch.empty(n, k, device="cuda")}
    x = (np.random.default_rng(seed).standard_normal((c["n"], c["k"]), dtype=np.float32) * np.float32(0.02))
    return {"kind": kind, "t": TYPES[c["type"]], "x": x}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        s = _stream()
        return [lin.forward(state["x"], m=state["m"], x_dtype=state["xd"], y=y, y_dtype=state["yd"], stream=s) for lin, y in state["stack"]]
    if kind == "decode":
        lib, s = state["lib"], _stream()
        if state["recording"]:
            pm.check(lib.pmetal_hip_replay(state["recording"].handle, s))
        else:
            for descs, count in state["calls"]:
                pm.check(lib.pmetal_hip_qgemv_batch(descs, count, s))
        return state["out"]
    if kind == "gemm_batches":
        lib, s = state["lib"], _stream()
        for descs, count, k, x in state["calls"]:
            pm.check(lib.pmetal_hip_qgemm_batch(descs, count, k, x.data_ptr(), state["xd"], state["m"], s))
        return state["outs"]
    if kind == "quantize":
        pm.check(state["lib"].pmetal_hip_quantize_batch_dev(state["descs"], len(state["descs"]), _stream()), "quantize")
        return state["outs"]
    if kind == "dequantize":
        blocks, out = state["blocks"], state["out"]
        pm.check(state["lib"].pmetal_hip_dequantize_dev(state["t"], blocks.data_ptr(), blocks.numel(), out.data_ptr(), out.numel(), state["order"], _stream()))
        return out
    blocks = pm.quantize(state["x"], state["t"])
    return [blocks, pm.dequantize(blocks, state["t"], state["x"].shape)]


# ---- what a pass cannot do without ----
def _matmul_work(t, n, k, m, xb, yb):
    return {"bytes": _nbytes(t, n * k) + m * k * xb + m * n * yb, "flops": 2 * m * n * k}


def _add(parts):
    return {"bytes": sum(p["bytes"] for p in parts), "flops": sum(p["flops"] for p in parts)}


def work(case):
    c, kind = case, case["kind"]
    size = {"bf16": 2, "f32": 4}
    if kind == "linear":
        one = _matmul_work(c["type"], c["n"], c["k"], c["m"], 0, size[c["y"]])
        return {"bytes": c["layers"] * one["bytes"] + c["m"] * c["k"] * size[c["x"]], "flops": c["layers"] * one["flops"]}
    if kind == "pair":
        one = _matmul_work(c["type"], c["n"], c["k"], c["m"], 0, size[c["y"]])
        return {"bytes": 2 * c["layers"] * one["bytes"] + c["m"] * c["k"] * size[c["x"]], "flops": 2 * c["layers"] * one["flops"]}
    if kind in ("decode", "prefill"):
        layers, m, yb = (c["layers"], 1, 4) if kind == "decode" else (1, c["m"], 2)
        parts = []
        for tensors in _layer_tensors(c, layers):
            for group in GROUPS:
                for i, at in enumerate(group):
                    name, n, k = tensors[at]
                    parts.append(_matmul_work(_recipe(name, layers), n, k, m, 2 if i == 0 else 0, yb))
        if c.get("vocab"):
            parts.append(_matmul_work(_recipe("output.weight", layers), c["vocab"], c["hidden"], 1, 2, 4))
        return _add(parts)
    if kind == "quantize":
        # at the least a multiplication, a rounding and two clamps an element, and two sums of the scale search
        return _add([{"bytes": 4 * n * k + _nbytes(_recipe(name, c["layers"]), n * k), "flops": 8 * n * k} for layer in _layer_tensors(c, c["layers"]) for name, n, k in layer])
    elements = c["n"] * c["k"]
    if kind == "dequantize":
        return {"bytes": 4 * elements + _nbytes(c["type"], elements), "flops": 2 * elements}
    return {"bytes": 2 * (4 * elements + _nbytes(c["type"], elements)), "flops": 4 * elements}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quantize", "dequantize", "host_codec"):
        return "exact"
    if kind == "decode" or (kind == "linear" and case["m"] == 1):
        return {"rel": 1e-5}
    if kind == "prefill" or case["y"] == "bf16":
        return {"rel": 7e-3}  # a result rounded to bf16 is 1.7e-3 from the product in 64 bits
    return {"rel": 1e-5} if case["x"] == "bf16" else {"rel": 1e-3}  # f32 activations of a matrix product are taken at f16's eleven bits
