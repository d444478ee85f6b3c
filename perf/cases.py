"""The work this framework is timed on: packed-ternary linear layers in every way a program
uses them, and the codecs that make their weights.

A case is a dict of plain values; ``kind`` says which path it takes:

* ``linear``  -- ``t81lib_amd.nn.Linear`` in eval mode under ``no_grad``, called eagerly;
* ``step``    -- the four projections of a few decoder layers (``nn.Linear``) as one captured
  decode step, replayed;
* ``int8``    -- ``ops.ternary_matmul`` with int8 activations (exact int32 results);
* ``grad``    -- a frozen eval-mode ``nn.Linear`` inside a differentiated program: forward and
  the gradients of its input and bias;
* ``train``   -- ``nn.Linear`` in train mode (quantization-aware): forward and all gradients;
* ``pack``    -- ``TernaryTensor.update_from_float``: new float weights into packed limbs;
* ``gguf``    -- a GGUF tensor payload: ``gguf.quantize_tensor`` and ``gguf.dequantize_tensor``.

Layer sizes are those of this repository's benchmark (the Llama-3-8B and Phi-3 projections) and
odd ones beside them.
"""

from __future__ import annotations

import math

import torch

from t81lib_amd import gguf, nn, ops, tensor

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
LAYER_THRESHOLD = 0.45  # nn.Linear's own default


def listed():
    return [
        # One token through the smallest projection, called from Python: the latency of a call.
        {"name": "linear_1x3072x3072_bf16", "kind": "linear", "m": 1, "k": 3072, "n": 3072,
         "dtype": "bf16", "bias": False},
        # Greedy decoding of one sequence: every projection of four decoder layers, captured
        # once and replayed per token, as the benchmark's stack decodes.
        {"name": "step_1_bf16", "kind": "step", "m": 1, "hidden": 4096, "qkv": 6144,
         "ffn": 14336, "layers": 4, "dtype": "bf16"},
        # The same step for a batch of 32 sequences.
        {"name": "step_32_bf16", "kind": "step", "m": 32, "hidden": 4096, "qkv": 6144,
         "ffn": 14336, "layers": 4, "dtype": "bf16"},
        # A small batch with float32 activations (a float32 module's default) and a bias.
        {"name": "linear_48x4096x14336_f32", "kind": "linear", "m": 48, "k": 4096, "n": 14336,
         "dtype": "f32", "bias": True},
        # A ragged prompt: a token count no tile divides.
        {"name": "linear_777x3072x9216_bf16", "kind": "linear", "m": 777, "k": 3072, "n": 9216,
         "dtype": "bf16", "bias": True},
        # A long prompt through the widest projection.
        {"name": "linear_2048x4096x28672_bf16", "kind": "linear", "m": 2048, "k": 4096,
         "n": 28672, "dtype": "bf16", "bias": False},
        # A prompt with float32 activations through the deepest projection.
        {"name": "linear_2048x14336x4096_f32", "kind": "linear", "m": 2048, "k": 14336,
         "n": 4096, "dtype": "f32", "bias": True},
        # Activations already quantized to int8: exact integer results.
        {"name": "int8_1536x4096x6144", "kind": "int8", "m": 1536, "k": 4096, "n": 6144},
        # A frozen ternary layer under autograd (adapters, prompts or layers below it train).
        {"name": "grad_1024x4096x14336_f32", "kind": "grad", "m": 1024, "k": 4096, "n": 14336,
         "dtype": "f32", "bias": True},
        # Quantization-aware training of one layer.
        {"name": "train_2048x4096x4096_f32", "kind": "train", "m": 2048, "k": 4096, "n": 4096,
         "dtype": "f32", "bias": True},
        # Weights that changed are packed again (conversion, and each forward after a step).
        {"name": "pack_8192x3072_f32", "kind": "pack", "n": 8192, "k": 3072, "dtype": "f32",
         "threshold": 0.45},
        # One tensor of a GGUF file, written and read back.
        {"name": "gguf_8192x3072_TQ1_0", "kind": "gguf", "n": 8192, "k": 3072,
         "quant": "TQ1_0", "threshold": 0.45},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _features(rng, lo, hi):
    """A layer dimension: mostly a multiple of 64 as models have them, else any number."""
    v = _log_int(rng, lo, hi)
    return max(lo, min(hi, v // 64 * 64)) if rng.random() < 0.7 else v


def _mnk(rng, m_lo, m_hi, most):
    """Tokens, inputs and outputs whose product stays within ``most``."""
    while True:
        m, k, n = _log_int(rng, m_lo, m_hi), _features(rng, 512, 14336), _features(rng, 512, 28672)
        if m * k * n <= most:
            return m, k, n


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "step", "int8", "grad", "train",
                       "pack", "gguf"])
    if kind == "linear":
        dtype = rng.choice(["bf16", "bf16", "f32"])
        m, k, n = _mnk(rng, 1, 4096, 2048 * 4096 * (28672 if dtype == "bf16" else 14336))
        return {"kind": kind, "m": m, "k": k, "n": n, "dtype": dtype, "bias": rng.random() < 0.5}
    if kind == "step":
        hidden = _features(rng, 1024, 4096)
        return {"kind": kind, "m": _log_int(rng, 1, 32), "hidden": hidden,
                "qkv": _features(rng, hidden, 2 * hidden), "ffn": _features(rng, 2048, 14336),
                "layers": rng.randint(2, 4), "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "int8":
        m, k, n = _mnk(rng, 1, 4096, 2048 * 4096 * 14336)
        return {"kind": kind, "m": m, "k": k, "n": n}
    if kind == "grad":
        m, k, n = _mnk(rng, 16, 4096, 1024 * 4096 * 14336)
        return {"kind": kind, "m": m, "k": k, "n": n, "dtype": rng.choice(["f32", "bf16"]),
                "bias": rng.random() < 0.5}
    if kind == "train":
        m, k, n = _mnk(rng, 64, 4096, 2048 * 4096 * 4096)
        return {"kind": kind, "m": m, "k": k, "n": n, "dtype": rng.choice(["f32", "f32", "bf16"]),
                "bias": rng.random() < 0.5}
    k, n = _features(rng, 256, 14336), _features(rng, 256, 14336)
    if kind == "pack":
        return {"kind": kind, "n": n, "k": k, "dtype": rng.choice(["f32", "bf16", "f16"]),
                "threshold": rng.choice([0.45, 0.5])}
    return {"kind": kind, "n": n, "k": k, "quant": rng.choice(["TQ1_0", "TQ2_0"]),
            "threshold": rng.choice([0.0, 0.45, 0.5])}


# ------------------------------------------------------------------------------ inputs --

def _gen(seed):
    return torch.Generator("cuda").manual_seed(seed)


def _randn(g, *shape, dtype=torch.float32, std=1.0):
    t = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, std, generator=g)
    return t if dtype == torch.float32 else t.to(dtype)


def _weight(g, n, k):
    """Weights in units of their standard deviation: at the default threshold about a third
    of the trits are zero, as in a ternary network."""
    return _randn(g, n, k)


def _acts(g, m, k, dtype):
    """Normal activations with one in a hundred ten times as large, as hidden states have."""
    x = _randn(g, m, k)
    x.mul_(torch.where(torch.rand((m, k), device="cuda", generator=g) < 0.01, 10.0, 1.0))
    return x.to(dtype)


def _inputs(case, seed):
    """The tensors a program holds before the call, in the order they are drawn."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "step":
        h, f, m = case["hidden"], case["ffn"], case["m"]
        dtype = DTYPES[case["dtype"]]
        shapes = [(h, case["qkv"]), (h, h), (h, 2 * f), (f, h)]
        for _ in range(case["layers"]):
            for k, n in shapes:
                yield _weight(g, n, k), _acts(g, m, k, dtype)
        return
    if kind in ("linear", "grad"):
        yield _weight(g, case["n"], case["k"])
        yield _acts(g, case["m"], case["k"], DTYPES[case["dtype"]])
        yield _randn(g, case["n"]) if case["bias"] else None
        if kind == "grad":
            yield _randn(g, case["m"], case["n"])
        return
    if kind == "train":
        dtype = DTYPES[case["dtype"]]
        yield _randn(g, case["n"], case["k"], dtype=dtype, std=0.02)
        yield _randn(g, case["m"], case["k"], dtype=dtype)
        yield _randn(g, case["n"], dtype=dtype) if case["bias"] else None
        yield _randn(g, case["m"], case["n"], dtype=dtype)
        return
    if kind == "int8":
        yield _weight(g, case["n"], case["k"])
        yield torch.randint(-127, 128, (case["m"], case["k"]), dtype=torch.int8, device="cuda",
                            generator=g)
        return
    if kind == "pack":
        yield _randn(g, case["n"], case["k"], dtype=DTYPES[case["dtype"]])
        return
    yield _randn(g, case["n"], case["k"])  # gguf


def _eval_layer(w, bias):
    n, k = w.shape
    layer = nn.Linear(k, n, bias=bias is not None, device="meta").to_empty(device="cuda")
    layer.weight = torch.nn.Parameter(w, requires_grad=False)
    if bias is not None:
        layer.bias = torch.nn.Parameter(bias)
    return layer.eval()


def prepare(case, seed):
    kind = case["kind"]
    it = _inputs(case, seed)
    if kind == "step":
        layers, xs = [], []
        with torch.no_grad():
            for w, x in it:
                layer = _eval_layer(w, None)
                layer(x)  # packs the weight
                layers.append(layer)
                xs.append(x)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                ys = [layer(x) for layer, x in zip(layers, xs)]
        return {"kind": kind, "graph": graph, "ys": ys, "layers": layers, "xs": xs}
    if kind == "linear":
        w, x, bias = it
        layer = _eval_layer(w, bias)
        with torch.no_grad():
            layer(x[:1])  # packs the weight
        return {"kind": kind, "layer": layer, "x": x}
    if kind == "grad":
        w, x, bias, g = it
        layer = _eval_layer(w, bias)
        x.requires_grad_(True)
        layer(x[:1]).sum().backward()  # packs the weight and its transpose
        return {"kind": kind, "layer": layer, "x": x, "g": g}
    if kind == "train":
        w, x, bias, g = it
        n, k = w.shape
        layer = nn.Linear(k, n, bias=bias is not None, device="meta").to_empty(device="cuda")
        layer.weight = torch.nn.Parameter(w)
        if bias is not None:
            layer.bias = torch.nn.Parameter(bias)
        return {"kind": kind, "layer": layer.train(), "x": x.requires_grad_(True), "g": g}
    if kind == "int8":
        w, x = it
        packed = tensor.TernaryTensor.from_float(w, threshold=LAYER_THRESHOLD).packed
        return {"kind": kind, "w": packed, "x": x, "k": case["k"]}
    if kind == "pack":
        (w,) = it
        held = tensor.TernaryTensor.from_float(torch.zeros_like(w), threshold=case["threshold"])
        return {"kind": kind, "w": w, "held": held}
    (w,) = it
    return {"kind": kind, "w": w, "quant": case["quant"], "threshold": case["threshold"]}


def run(state):
    kind = state["kind"]
    if kind == "step":
        state["graph"].replay()
        return state["ys"]
    if kind == "linear":
        with torch.no_grad():
            return state["layer"](state["x"])
    if kind in ("grad", "train"):
        layer, x = state["layer"], state["x"]
        x.grad = None
        layer.zero_grad(set_to_none=True)
        y = layer(x)
        y.backward(state["g"])
        out = {"y": y.detach(), "dx": x.grad}
        if kind == "train":
            out["dw"] = layer.weight.grad
        if layer.bias is not None:
            out["db"] = layer.bias.grad
        return out
    if kind == "int8":
        return ops.ternary_matmul(state["x"], state["w"], state["k"])
    if kind == "pack":
        state["held"].update_from_float(state["w"])
        return state["held"].packed
    payload = gguf.quantize_tensor(state["w"], state["quant"], state["threshold"])
    return payload, gguf.dequantize_tensor(payload, state["w"].shape, state["quant"])


# ---------------------------------------------------------------------------- the bounds --

SIZE = {"f32": 4, "bf16": 2, "f16": 2}


def _limb_bytes(n, k):
    return 16 * n * ((k + 47) // 48)


def _linear_bytes(m, n, k, s, bias):
    return _limb_bytes(n, k) + s * m * k + 4 * m * n + (4 * n if bias else 0)


def work(case):
    kind, n, k, m = case["kind"], case.get("n"), case.get("k"), case.get("m")
    if kind == "step":
        h, f, s = case["hidden"], case["ffn"], SIZE[case["dtype"]]
        shapes = [(h, case["qkv"]), (h, h), (h, 2 * f), (f, h)]
        return {"bytes": case["layers"] * sum(_linear_bytes(m, b, a, s, False) for a, b in shapes),
                "flops": case["layers"] * sum(2.0 * m * a * b for a, b in shapes)}
    if kind == "linear":
        return {"bytes": _linear_bytes(m, n, k, SIZE[case["dtype"]], case["bias"]),
                "flops": 2.0 * m * n * k}
    if kind == "int8":
        return {"bytes": _linear_bytes(m, n, k, 1, False), "flops": 2.0 * m * n * k}
    if kind == "grad":  # forward, and the transposed product of the backward
        s = SIZE[case["dtype"]]
        return {"bytes": _linear_bytes(m, n, k, s, case["bias"]) + 4 * m * n + s * m * k
                + _limb_bytes(k, n) + (4 * n if case["bias"] else 0), "flops": 4.0 * m * n * k}
    if kind == "train":  # x, w, g in; y, dx, dw out; three products
        s = SIZE[case["dtype"]]
        return {"bytes": s * (2 * m * k + 2 * n * k + 2 * m * n + (2 * n if case["bias"] else 0)),
                "flops": 6.0 * m * n * k}
    if kind == "pack":
        return {"bytes": SIZE[case["dtype"]] * n * k + _limb_bytes(n, k), "flops": 0.0}
    payload = n * gguf.row_bytes(k, case["quant"])
    return {"bytes": 2 * 4 * n * k + 2 * payload, "flops": 0.0}


def tolerance(case):
    kind = case["kind"]
    if kind in ("int8", "pack", "gguf"):
        return "exact"
    if kind == "train":
        # float32: the library's sums are up to 8e-7 from 64 bits (the weight gradient's);
        # bfloat16: results rounded to it (1.7e-3)
        return {"rel": 4e-6, "max": 1e-4} if case["dtype"] == "f32" else {"rel": 7e-3, "max": 0.05}
    if kind == "grad" and case["dtype"] == "bf16":  # dx is rounded to the input's bf16
        return {"rel": 7e-3, "max": 0.05}
    if case["dtype"] == "bf16":  # exact products, float32 sums: up to 1e-7 from 64 bits
        return {"rel": 5e-7, "max": 1e-5}
    return {"rel": 1e-5, "max": 1e-4}  # float32 as two bfloat16 values: 2.6e-6


# ------------------------------------------------------------------------- 64-bit results --

def _trits(w, threshold):
    """Ternary decisions are made in float32 (``w >= thr``), as the packer's are."""
    t = torch.tensor(threshold, dtype=torch.float32, device=w.device)
    w = w.float()
    return (w >= t).double() - (w <= -t).double()


def _exact_gguf(w, quant, threshold):
    n, k = w.shape
    nb = (k + 255) // 256
    blocks = torch.nn.functional.pad(w, (0, nb * 256 - k)).reshape(n, nb, 256)
    d = blocks.abs().amax(dim=2, keepdim=True)
    inv = torch.where(d == 0, torch.zeros_like(d), 1.0 / d)
    v = blocks * inv
    if threshold > 0:
        thr = torch.tensor(threshold, dtype=torch.float32, device=w.device)
        t = torch.where(v.abs() >= thr, torch.sign(v), torch.zeros_like(v))
    else:
        t = torch.where(v >= 0, torch.floor(v + 0.5), torch.ceil(v - 0.5)).clamp(-1, 1)
    out = t.double() * d.half().double()
    return out.reshape(n, nb * 256)[:, :k].contiguous()


def exact(case, seed):
    kind = case["kind"]
    it = _inputs(case, seed)
    if kind == "step":
        return [x.double() @ _trits(w, LAYER_THRESHOLD).T for w, x in it]
    if kind == "int8":
        w, x = it
        return (x.double() @ _trits(w, LAYER_THRESHOLD).T).to(torch.int32)
    if kind == "pack":
        return None  # bytes
    if kind == "gguf":
        (w,) = it
        return None, _exact_gguf(w, case["quant"], case["threshold"])
    if kind == "linear":
        w, x, bias = it
        y = x.double() @ _trits(w, LAYER_THRESHOLD).T
        return y + bias.double() if bias is not None else y
    if kind == "grad":
        w, x, bias, g = it
        t = _trits(w, LAYER_THRESHOLD)
        y = x.double() @ t.T
        out = {"y": y + bias.double() if bias is not None else y, "dx": g.double() @ t}
        if bias is not None:
            out["db"] = g.double().sum(0)
        return out
    # train: the layer's scale is max |w| on its first step; w / s and the two comparisons
    # are decided in the weight's own type
    w, x, bias, g = it
    s = w.abs().amax().clamp(min=1e-6).float()
    u = w / s
    q = torch.where(u.abs() >= LAYER_THRESHOLD, torch.sign(u), torch.zeros_like(u))
    t, scale, g64 = (q * s).double(), s.double(), g.double()
    y = x.double() @ t.T
    dw = (g64.T @ x.double()) * scale
    half = u.abs() < 0.5
    out = {"y": y + bias.double() if bias is not None else y, "dx": g64 @ t,
           "dw": torch.where(half, 2.0 * dw, torch.zeros_like(dw)) / scale}
    if bias is not None:
        out["db"] = g64.sum(0)
    return out
