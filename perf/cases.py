"""The measured workloads: what a program that uses this library has it do,
through the public Python entry points (funasrnet_amd.hip) over the C ABI.

The library stands behind a speech recogniser: an FP32 audio encoder (its
projections, feed-forward pairs and attention), whose output rows a Q8_0
Qwen3 decoder takes as its prefix (prefill) before it generates text greedily
(decode), one recording at a time or many in lock step. Layers are called on
device buffers (torch tensors, as a program that keeps its activations on the
GPU has them) or on host buffers where a caller of the backend seam has them
there. Weights are random of the real shapes; activations are N(0, 1), which
is what normalised rows are.

Import torch before the library is loaded (this file does): the library then
binds to the HIP runtime that torch brought, and both share the device.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from funasrnet_amd import model
from funasrnet_amd.hip import HipBackend, HipDecoder, HipFloatWeight, HipWeight

_shared: dict = {}


def listed() -> list:
    return [
        # One token's q projection: the smallest call, one short kernel.
        {"name": "q8_token", "kind": "q8", "frames": 1, "cols": 1024, "rows": 2048},
        # The fused q/k/v projection of a 20-second prefix.
        {"name": "q8_prefix", "kind": "q8", "frames": 375, "cols": 1024, "rows": 4096},
        # The decoder with its original FP32 weights: one token's gate rows.
        {"name": "f32_token", "kind": "f32", "frames": 1, "cols": 1024, "rows": 3072, "bias": False},
        # The encoder's first layer: seven stacked 80-bin frames to q/k/v, 20 s of audio.
        {"name": "f32_first_layer", "kind": "f32", "frames": 333, "cols": 560, "rows": 1536, "bias": True},
        # The feed-forward's wide projection, one 60-second segment.
        {"name": "f32_segment", "kind": "f32", "frames": 1000, "cols": 512, "rows": 2048, "bias": True},
        # The feed-forward's way back, several segments together.
        {"name": "f32_long", "kind": "f32", "frames": 4000, "cols": 2048, "rows": 512, "bias": True},
        # The encoder's self-attention, one 60-second segment and the longest the entry point takes.
        {"name": "attention_segment", "kind": "attention", "frames": 1000, "width": 512, "heads": 4},
        {"name": "attention_longest", "kind": "attention", "frames": 4096, "width": 512, "heads": 4},
        # The encoder's feed-forward pair from and to host memory, as the seam's callers have it.
        {"name": "ffn_host", "kind": "ffn", "frames": 500, "width": 512, "hidden": 2048},
        # Time to the first token of a 20-second recording.
        {"name": "prefill", "kind": "prefill", "rows": 375},
        # Greedy text of one recording after a 150-row prefix.
        {"name": "decode", "kind": "decode", "sessions": 1, "prefix": 150, "steps": 32},
        # Sixteen recordings in lock step, as the server runs them.
        {"name": "decode_sessions", "kind": "decode", "sessions": 16, "prefix": 150, "steps": 32},
    ]


def _between(rng, low: int, high: int) -> int:
    """Log-uniform whole number of [low, high]."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng) -> dict:
    kind = rng.choice(["q8", "q8", "f32", "f32", "f32", "attention", "attention", "ffn", "prefill", "decode", "decode"])
    if kind == "q8":
        # A token, a few sessions' rows, or a prefix; widths of whole Q8_0
        # blocks, mostly the multiples of 128 that model widths are. The
        # lm_head's many rows only for a token.
        frames = rng.choice([1, _between(rng, 2, 16), _between(rng, 17, 750)])
        cols = 128 * _between(rng, 4, 24) if rng.random() < 0.75 else 32 * _between(rng, 16, 96)
        return {"kind": kind, "frames": frames, "cols": cols, "rows": _between(rng, 256, 152000 if frames == 1 else 6144)}
    if kind == "f32":
        frames = rng.choice([1, _between(rng, 2, 32), _between(rng, 33, 4000), _between(rng, 33, 4000)])
        cols = 4 * _between(rng, 64, 512) if rng.random() < 0.8 else _between(rng, 256, 2048)
        return {"kind": kind, "frames": frames, "cols": cols, "rows": _between(rng, 256, 3072 if frames == 1 else 2048),
                "bias": rng.random() < 0.7}
    if kind == "attention":
        size = rng.choice([128, 128, 64, 96])
        heads = rng.choice([4, 8]) if size < 128 else 4
        return {"kind": kind, "frames": _between(rng, 160, 4096 if size * heads <= 512 and size != 96 else 1200),
                "width": size * heads, "heads": heads}
    if kind == "ffn":
        return {"kind": kind, "frames": _between(rng, 20, 1500), "width": rng.choice([320, 512, 560]), "hidden": rng.choice([1024, 2048])}
    if kind == "prefill":
        return {"kind": kind, "rows": _between(rng, 8, 750)}
    if rng.random() < 0.5:
        return {"kind": kind, "sessions": rng.randint(2, 16), "prefix": _between(rng, 40, 250), "steps": rng.randint(8, 32)}
    return {"kind": kind, "sessions": 1, "prefix": _between(rng, 20, 2048), "steps": rng.randint(8, 32)}


# ---- What a program holds ------------------------------------------------------


def _backend() -> HipBackend:
    if "backend" not in _shared:
        _shared["backend"] = HipBackend(0)
    return _shared["backend"]


def _weights() -> model.DecoderWeights:
    if "weights" not in _shared:
        _shared["weights"] = model.synthetic(model.QWEN3_0_6B, seed=0)
    return _shared["weights"]


def _decoder() -> HipDecoder:
    """The loaded model: recordings are sessions over its device weights."""
    if "decoder" not in _shared:
        _shared["decoder"] = HipDecoder(_backend(), _weights(), capacity=64)
    return _shared["decoder"]


def _normal(gen, *shape, scale: float = 1.0) -> torch.Tensor:
    return torch.randn(*shape, generator=gen, device="cuda") * scale


def _inputs(case: dict, seed: int) -> dict:
    """The case's inputs as torch tensors on the GPU, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "q8":
        rows, cols = case["rows"], case["cols"]
        return {"x": _normal(gen, case["frames"], cols),
                "q": torch.randint(-127, 128, (rows, cols), generator=gen, device="cuda", dtype=torch.int8),
                "s": (_normal(gen, rows, cols // 32, scale=0.02 / 127).abs()).half().float()}
    if kind == "f32":
        rows, cols = case["rows"], case["cols"]
        return {"x": _normal(gen, case["frames"], cols), "w": _normal(gen, rows, cols, scale=cols**-0.5),
                "b": _normal(gen, rows, scale=0.1) if case["bias"] else None}
    if kind == "attention":
        return {k: _normal(gen, case["frames"], case["width"]) for k in ("q", "k", "v")}
    if kind == "ffn":
        width, hidden = case["width"], case["hidden"]
        return {"x": _normal(gen, case["frames"], width), "w1": _normal(gen, hidden, width, scale=width**-0.5),
                "b1": _normal(gen, hidden, scale=0.1), "w2": _normal(gen, width, hidden, scale=hidden**-0.5),
                "b2": _normal(gen, width, scale=0.1)}
    rows = case["rows"] if kind == "prefill" else case["prefix"]
    count = case["sessions"] if kind == "decode" else 1
    return {"x": _normal(gen, count, rows, model.QWEN3_0_6B.width)}


def prepare(case: dict, seed: int) -> dict:
    backend, kind = _backend(), case["kind"]
    v = _inputs(case, seed)
    state = {"case": case, "backend": backend}
    if kind == "q8":
        state["weight"] = HipWeight(backend, model.Q8Tensor("w", v["q"].cpu().numpy(), v["s"].cpu().numpy()))
        state["x"] = v["x"]
        state["codes"] = torch.empty(v["x"].shape, dtype=torch.int8, device="cuda")
        state["scales"] = torch.empty((case["frames"], case["cols"] // 32), device="cuda")
        state["out"] = torch.empty((case["frames"], case["rows"]), device="cuda")
    elif kind == "f32":
        state["weight"] = HipFloatWeight(backend, v["w"].cpu().numpy())
        state["x"], state["b"] = v["x"], v["b"]
        state["out"] = torch.empty((case["frames"], case["rows"]), device="cuda")
    elif kind == "attention":
        state.update(v, out=torch.empty_like(v["q"]))
    elif kind == "ffn":
        state.update({k: t.cpu().numpy() for k, t in v.items()}, out=np.empty((case["frames"], case["width"]), np.float32))
        # The seam keeps a device copy of each weight from its first use on.
        backend.float_weight(state["w1"])
        backend.float_weight(state["w2"])
    elif kind == "prefill":
        state["x"] = v["x"][0].cpu().numpy()
        state["decoder"] = _decoder().session(case["rows"] + 8)
    else:
        x = v["x"].cpu().numpy()
        state["last"] = [np.ascontiguousarray(row[-1:]) for row in x]
        state["decoders"] = [_decoder().session(case["prefix"] + case["steps"] + 8) for _ in x]
        for d, row in zip(state["decoders"], x):
            d.decode(row, case["prefix"], output_logits=False)
    return state


def run(state: dict):
    case, backend, kind = state["case"], state["backend"], state["case"]["kind"]
    if kind == "q8":
        x, out = state["x"], state["out"]
        codes, scales = state["codes"], state["scales"]
        backend.quantize_device(x.data_ptr(), x.numel(), codes.data_ptr(), scales.data_ptr())
        backend.gemv_device(codes.data_ptr(), scales.data_ptr(), case["frames"], state["weight"], out.data_ptr())
        return {"out": out, "scales": scales, "codes": codes}
    if kind == "f32":
        b, out = state["b"], state["out"]
        backend.linear_device(state["x"].data_ptr(), case["frames"], state["weight"],
                              None if b is None else b.data_ptr(), out.data_ptr())
        return out
    if kind == "attention":
        out = state["out"]
        backend.attention_device(state["q"].data_ptr(), state["k"].data_ptr(), state["v"].data_ptr(), case["frames"],
                                 case["width"], case["heads"], out.data_ptr())
        return out
    if kind == "ffn":
        backend.try_relu_projection(state["x"], case["frames"], state["w1"], state["b1"], state["w2"], state["b2"],
                                    state["out"])
        return state["out"]
    if kind == "prefill":
        d = state["decoder"]
        d.reset()
        return d.decode(state["x"], case["rows"])
    # The prefix is cached; its last row again gives the first logits, the
    # text follows, and one more step returns the logits after it.
    first = []
    for d, row in zip(state["decoders"], state["last"]):
        d.set_position(case["prefix"] - 1)
        first.append(d.decode(row, 1))
    if len(first) == 1:
        d = state["decoders"][0]
        tokens = d.generate(case["steps"])[None]
    else:
        tokens = HipDecoder.generate_sessions(state["decoders"], case["steps"])
    d = state["decoders"][0]
    return {"first": first, "tokens": tokens, "last": d.decode(d.embed(tokens[0, -1:]), 1)}


# ---- What the work cannot do without -----------------------------------------------


def _layers_flops(positions_seen: float, rows: int) -> float:
    """Multiply-adds x 2 of the decoder layers over `rows` rows that see
    `positions_seen` positions in all."""
    c = model.QWEN3_0_6B
    matrix = (c.weight_bytes_per_token() * 32 // 34) - c.vocab * c.width
    return 2.0 * matrix * rows + 4.0 * c.layers * c.q_width * positions_seen


def work(case: dict) -> dict:
    kind, c = case["kind"], model.QWEN3_0_6B
    if kind == "q8":
        f, n, k = case["frames"], case["rows"], case["cols"]
        return {"bytes": n * k * 34 / 32 + 4 * f * k + f * k * 36 / 32 + 4 * f * n, "flops": 2.0 * f * n * k}
    if kind == "f32":
        f, n, k = case["frames"], case["rows"], case["cols"]
        return {"bytes": 4.0 * (n * k + f * k + f * n + (n if case["bias"] else 0)), "flops": 2.0 * f * n * k}
    if kind == "attention":
        f, w = case["frames"], case["width"]
        return {"bytes": 16.0 * f * w, "flops": 4.0 * f * f * w}
    if kind == "ffn":
        f, w, h = case["frames"], case["width"], case["hidden"]
        return {"bytes": 4.0 * (2 * f * w + 2 * w * h + w + h), "flops": 4.0 * f * w * h}
    head_flops, kv_row = 2.0 * c.vocab * c.width, 4 * c.layers * c.kv_width
    if kind == "prefill":
        t = case["rows"]
        return {"bytes": float(c.weight_bytes_per_token()) + kv_row * t + 4 * t * c.width + 4 * c.vocab,
                "flops": _layers_flops(t * (t + 1) / 2, t) + head_flops}
    # Every step reads the weights once for all sessions; the prefix's last
    # row is decoded for each session alone, and one more step for the first.
    n, p, s = case["sessions"], case["prefix"], case["steps"]
    cached = n * p + n * sum(p + 1 + i for i in range(s)) + p + s + 1
    return {"bytes": float(c.weight_bytes_per_token()) * (n + s + 1) + kv_row * cached,
            "flops": _layers_flops(cached, n * (s + 1) + 1) + head_flops * (n * (s + 1) + 1)}


def tolerance(case: dict):
    """Q8_0 paths fix the order of every sum (the reference's), so any
    implementation gives the same bits; FP32 ones may add in any order."""
    kind = case["kind"]
    if kind in ("q8", "prefill", "decode"):
        return "exact"
    # Measured against 64 bits: 1e-7 to 8e-7 for the projections (sums of 256
    # to 2048 products), 5e-7 for the feed-forward pair, 7e-7 for attention.
    return {"rel": 4e-6, "max": 1e-4}


# ---- The same in 64 bits ------------------------------------------------------------


def _quantized(x: torch.Tensor) -> torch.Tensor:
    """Rows after Q8_0 rounding of each 32 values (scale amax / 127, halves away from zero)."""
    blocks = x.reshape(-1, 32).float()
    d = blocks.abs().amax(1, keepdim=True) / 127
    v = blocks * torch.where(d == 0, torch.zeros_like(d), 1 / d)
    codes = (torch.floor(v.abs().double() + 0.5) * torch.sign(v)).clamp(-127, 127)
    return (codes * d.double()).reshape(x.shape)


def _matrix(t: model.Q8Tensor) -> torch.Tensor:
    q = torch.from_numpy(t.quantized).cuda().double().reshape(t.rows, -1, 32)
    return (q * torch.from_numpy(t.scales).cuda().double()[..., None]).reshape(t.rows, -1)


def _attention64(q, k, v, heads: int, causal: bool) -> torch.Tensor:
    """[rows, heads * size] of each head's softmax(q k^T / sqrt(size)) v."""
    size, out = q.shape[1] // heads, []
    group = q.shape[1] // k.shape[1]
    for h in range(heads):
        a = slice(h * size, (h + 1) * size)
        b = slice(h // group * size, (h // group + 1) * size)
        s = q[:, a] @ k[:, b].T / math.sqrt(size)
        if causal:
            s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), -math.inf)
        out.append(torch.softmax(s, 1) @ v[:, b])
    return torch.cat(out, 1)


def _logits64(x: torch.Tensor) -> torch.Tensor:
    """Logits of the last of the prefix rows x, from an empty cache."""
    w, c = _weights(), model.QWEN3_0_6B
    x = x.double()
    at = torch.arange(x.shape[0], device="cuda", dtype=torch.float64)[:, None]
    angle = at * c.rope_base ** (-torch.arange(0, c.head_size, 2, device="cuda", dtype=torch.float64) / c.head_size)
    cos, sin = torch.cos(angle)[:, None], torch.sin(angle)[:, None]

    def norm(v, scale):
        return v * torch.rsqrt(v.square().mean(-1, keepdim=True) + c.eps) * torch.from_numpy(scale).cuda().double()

    def heads(v, scale):
        v = norm(v.reshape(v.shape[0], -1, c.head_size), scale)
        a, b = v.chunk(2, -1)
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1).flatten(1)

    for layer in w.layers:
        h = _quantized(norm(x, layer.attn_norm))
        q, k = heads(h @ _matrix(layer.wq).T, layer.q_norm), heads(h @ _matrix(layer.wk).T, layer.k_norm)
        v = h @ _matrix(layer.wv).T
        x = x + _quantized(_attention64(q, k.half().double(), v.half().double(), c.heads, True)) @ _matrix(layer.wo).T
        h = _quantized(norm(x, layer.ffn_norm))
        g = h @ _matrix(layer.gate).T
        x = x + _quantized(g * torch.sigmoid(g) * (h @ _matrix(layer.up).T)) @ _matrix(layer.down).T
    return (_quantized(norm(x[-1:], w.output_norm)) @ _matrix(w.lm_head).T)[0]


def exact(case: dict, seed: int):
    v, kind = _inputs(case, seed), case["kind"]
    if kind == "q8":
        w = (v["q"].double().reshape(case["rows"], -1, 32) * v["s"].double()[..., None]).reshape(case["rows"], -1)
        scales = v["x"].double().reshape(case["frames"], -1, 32).abs().amax(2) / 127
        return {"out": _quantized(v["x"]) @ w.T, "scales": scales, "codes": None}
    if kind == "f32":
        out = v["x"].double() @ v["w"].double().T
        return out if v["b"] is None else out + v["b"].double()
    if kind == "attention":
        return _attention64(v["q"].double(), v["k"].double(), v["v"].double(), case["heads"], False)
    if kind == "ffn":
        hidden = torch.relu(v["x"].double() @ v["w1"].double().T + v["b1"].double())
        return (hidden @ v["w2"].double().T + v["b2"].double()).cpu().numpy()
    if kind == "prefill":
        return _logits64(v["x"][0]).cpu().numpy()
    if case["prefix"] > 512:
        return None
    return {"first": [_logits64(x).cpu().numpy() for x in v["x"]], "tokens": None, "last": None}
