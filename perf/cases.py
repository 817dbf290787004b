"""The work whose speed this library is measured by: decode, verification and
prefill products over packed-affine and dense F16 weights, called as a
program calls them (one command, its encodes, finish) through the `qmr`
binding.

Sizes are the decoder shapes that the repository's benchmark and tests use
(hidden 5120, MLP 17408, projections 5120x5120 and 12288x4096, a 151936-row
vocabulary), a small matrix, and ragged shapes. Weights and activations have
the benchmark's distributions: uniform codes, scales U(0.002, 0.02) for Q4
and U(1e-4, 2e-3) for Q8, biases near minus half the code range times the
scale, activations N(0, 1).

Weights, input and output buffers live on the device, as in a program that
decodes; a pass ends with the command's finish, and its outputs stay in their
device buffers unless the program needs them on the host (the vocabulary
head's logits, which it samples from).
"""
from __future__ import annotations

import functools
import math
import struct
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "qwen-mlx-runner_amd"))

import qmr  # noqa: E402

SUFFIX = {"f32": "", "bf16": "_bf16", "f16": "_f16meta"}
META_BYTES = {"f32": 4, "bf16": 2, "f16": 2}
EPS = 1e-6


# ---- the cases ----

def listed() -> list[dict]:
    return [
        # The smallest call: one small projection of one token, where the
        # command's own latency counts.
        {"name": "gemv_1024_b1", "kind": "product", "shape": "single", "rows": 1024, "cols": 1024,
         "bits": 4, "group": 64, "meta": "bf16", "batch": 1, "layers": 1},
        # Decode of one token: the fused MLP (norm + gate + up + SwiGLU, down
        # + residual) of four decoder layers in one command, each on a
        # residual stream of its own.
        {"name": "mlp_fused_b1", "kind": "mlp", "rows": 17408, "cols": 5120, "bits": 4, "group": 64,
         "meta": "bf16", "batch": 1, "layers": 4},
        # A verification block of three tokens: gate, up and down by the plain
        # block names, four layers in one command.
        {"name": "mlp_plain_b3", "kind": "product", "shape": "mlp", "rows": 17408, "cols": 5120,
         "bits": 4, "group": 64, "meta": "bf16", "batch": 3, "layers": 4},
        # Decode of one token through four 8-bit attention projections with
        # F16 metadata.
        {"name": "proj_q8_b1", "kind": "product", "shape": "single", "rows": 5120, "cols": 5120,
         "bits": 8, "group": 64, "meta": "f16", "batch": 1, "layers": 4},
        # The vocabulary head of one token, its logits read to the host.
        {"name": "head_b1", "kind": "head", "rows": 151936, "cols": 5120, "bits": 4, "group": 64,
         "meta": "bf16", "batch": 1},
        # A verification block over an unquantised (F16) MLP's up and down
        # matrices.
        {"name": "dense_f16_b3", "kind": "dense", "rows": 17408, "cols": 5120, "batch": 3},
        # Blocks in the other group size and FP32 metadata (the default
        # metadata mode), with ragged rows: four matrices, four tokens.
        {"name": "block_g32_f32_b4", "kind": "product", "shape": "single", "rows": 9001, "cols": 4160,
         "bits": 4, "group": 32, "meta": "f32", "batch": 4, "layers": 4},
        # Prefill of a short prompt: gate, up and down for 24 tokens.
        {"name": "prefill_mlp_24", "kind": "wide", "shape": "mlp", "rows": 17408, "cols": 5120, "bits": 4,
         "group": 64, "meta": "bf16", "batch": 24},
        # Prefill of a chunk: the same for 128 tokens.
        {"name": "prefill_mlp_128", "kind": "wide", "shape": "mlp", "rows": 17408, "cols": 5120, "bits": 4,
         "group": 64, "meta": "bf16", "batch": 128},
        # A large chunk with an odd number of tokens, FP32 metadata.
        {"name": "prefill_f32_211", "kind": "wide", "shape": "single", "rows": 12288, "cols": 4096, "bits": 4,
         "group": 64, "meta": "f32", "batch": 211},
        # Prefill through an 8-bit attention projection.
        {"name": "prefill_q8_64", "kind": "wide", "shape": "single", "rows": 5120, "cols": 5120, "bits": 8,
         "group": 64, "meta": "bf16", "batch": 64},
        # The embedding rows of a 96-token chunk, one encode for each token.
        {"name": "embed_96", "kind": "embed", "rows": 151936, "cols": 5120, "bits": 4, "group": 64,
         "meta": "bf16", "batch": 96},
    ]


def _log(rng, low: int, high: int, step: int = 1) -> int:
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, min(high, int(round(v / step)) * step))


def draw(rng) -> dict:
    """A case of the listed kinds: sizes over their whole ranges, ragged and
    odd ones among them, every format that its kind takes."""
    kind = rng.choice(["product", "product", "mlp", "wide", "wide", "wide", "dense", "head", "embed"])
    bits = rng.choice([4, 4, 8])
    group = rng.choice([64, 64, 32, 128])
    step = rng.choice([256, group])  # columns: whole groups, often a rounder number
    rows = _log(rng, 512, 24576, rng.choice([1, 16, 128]))
    cols = _log(rng, 1024, 17408, max(step, group))
    if rows * cols > 120_000_000:
        rows = 120_000_000 // cols
    if kind == "product":
        return {"kind": "product", "shape": "single", "rows": rows, "cols": cols, "bits": bits, "group": group,
                "meta": rng.choice(["f32", "bf16", "f16"]), "batch": rng.randint(1, 4), "layers": rng.randint(1, 4)}
    if kind == "mlp":  # formats that the fused launches take at every batch
        group = 64
        cols = _log(rng, 1024, 6144, 64)
        rows = min(cols * 3 + 64 * rng.randint(0, 30), 90_000_000 // cols) // 64 * 64
        return {"kind": "mlp", "rows": rows, "cols": cols, "bits": bits, "group": group,
                "meta": rng.choice(["f32", "bf16", "f16"]), "batch": rng.randint(1, 4),
                "layers": rng.randint(1, max(1, 480_000_000 // (3 * rows * cols * bits // 8)) if rows * cols > 20_000_000 else 4)}
    if kind == "wide":
        if bits == 8 or group != 64:
            rows = max(512, min(rows, 40_000_000 // cols))
        return {"kind": "wide", "shape": "single", "rows": rows, "cols": cols, "bits": bits, "group": group,
                "meta": rng.choice(["bf16", "bf16", "f32"]), "batch": _log(rng, 5, 256)}
    if kind == "dense":
        return {"kind": "dense", "rows": rows, "cols": _log(rng, 1024, 17408, 32) if rows <= 6144 else
                _log(rng, 1024, 5120, 32), "batch": rng.randint(1, 4)}
    if kind == "head":
        return {"kind": "head", "rows": _log(rng, 32000, 151936), "cols": _log(rng, 1024, 5120, group), "bits": 4,
                "group": group, "meta": rng.choice(["f32", "bf16"]), "batch": rng.randint(1, 2)}
    return {"kind": "embed", "rows": _log(rng, 32000, 151936), "cols": _log(rng, 1024, 5120, group), "bits": 4,
            "group": group, "meta": rng.choice(["f32", "bf16", "f16"]), "batch": _log(rng, 1, 96)}


# ---- inputs, made on the GPU from the seed alone ----

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _packed(g: torch.Generator, rows: int, cols: int, bits: int, group: int, meta: str):
    """(codes int32 [rows, cols*bits/32], scales, biases [rows, cols/group] as
    float32 holding values of the metadata type)."""
    w = torch.randint(-2**31, 2**31, (rows, cols * bits // 32), dtype=torch.int64, generator=g,
                      device="cuda").to(torch.int32)
    n = (rows, cols // group)
    low, high = (0.002, 0.02) if bits == 4 else (1e-4, 2e-3)
    s = torch.rand(n, generator=g, device="cuda") * (high - low) + low
    noise = torch.randn(n, generator=g, device="cuda") * (1e-3 if bits == 4 else 1e-4)
    # FP32 metadata holds a checkpoint's F16 values, expanded.
    kind = torch.bfloat16 if meta == "bf16" else torch.float16
    s = s.to(kind).float()
    b = (-float(2 ** (bits - 1)) * s + noise).to(kind).float()
    return w, s, b


def _normal(g: torch.Generator, *shape: int) -> torch.Tensor:
    return torch.randn(shape, generator=g, device="cuda")


def _inputs(case: dict, seed: int) -> dict:
    """The case's tensors: "matrices" (packed or dense) and what they are applied to."""
    g = _gen(seed)
    kind = case["kind"]
    rows, cols, batch = case["rows"], case["cols"], case["batch"]
    if kind == "dense":
        shapes = [(rows, cols), (cols, rows)]
        return {"matrices": [(_normal(g, *s) * (1 / math.sqrt(s[1]))).half() for s in shapes],
                "x": [_normal(g, batch, s[1]) for s in shapes]}
    fmt = (case["bits"], case["group"], case["meta"])
    if kind == "mlp":
        layers = [{"gate": _packed(g, rows, cols, *fmt), "up": _packed(g, rows, cols, *fmt),
                   "down": _packed(g, cols, rows, *fmt), "norm": 1 + 0.1 * _normal(g, cols),
                   "x": _normal(g, batch, cols)}
                  for _ in range(case["layers"])]
        return {"layers": layers}
    if kind == "embed":
        return {"matrices": [_packed(g, rows, cols, *fmt)],
                "tokens": torch.randint(0, rows, (batch,), generator=g, device="cuda").tolist()}
    layers = case.get("layers", 1)
    if case.get("shape") == "mlp":
        # Gate and up share the layer's input, down takes another.
        shapes, source = [], []
        for i in range(layers):
            shapes += [(rows, cols), (rows, cols), (cols, rows)]
            source += [2 * i, 2 * i, 2 * i + 1]
        widths = [cols, rows] * layers
    else:
        shapes, source, widths = [(rows, cols)] * layers, list(range(layers)), [cols] * layers
    return {"matrices": [_packed(g, *s, *fmt) for s in shapes], "source": source,
            "x": [_normal(g, batch, n) for n in widths]}


# ---- the program: device, resident buffers, the dispatches of one pass ----

@functools.lru_cache(maxsize=None)
def _gpu() -> qmr.Gpu:
    return qmr.Gpu("aligned", metadata="bf16")


def _upload(t: torch.Tensor) -> qmr.Buffer:
    return _gpu().upload_bytes(t.contiguous().cpu().numpy())


def _upload_meta(t: torch.Tensor, meta: str) -> qmr.Buffer:
    if meta == "f32":
        return _upload(t)
    return _upload(t.to(torch.bfloat16 if meta == "bf16" else torch.float16).view(torch.int16))


def _upload_packed(m, meta: str) -> list[qmr.Buffer]:
    w, s, b = m
    return [_upload(w), _upload_meta(s, meta), _upload_meta(b, meta)]


class DeviceOutputs(dict):
    """Output buffers by name. They stay on the device; looking at one copies
    it to the host."""

    def __getitem__(self, name):
        buffer, shape = super().__getitem__(name)
        return _gpu().read_f32(buffer, math.prod(shape)).reshape(shape)


def _call(name: str, buffers: list, params: list, offsets=None) -> tuple:
    return name, buffers, params, qmr.dispatch_layout(name, params)[1], offsets


def _eps_bits() -> int:
    return struct.unpack("<I", struct.pack("<f", EPS))[0]


def prepare(case: dict, seed: int) -> dict:
    t = _inputs(case, seed)
    gpu, kind = _gpu(), case["kind"]
    rows, cols, batch = case["rows"], case["cols"], case["batch"]
    calls, out = [], {}
    if kind == "dense":
        for i, (w, x) in enumerate(zip(t["matrices"], t["x"])):
            r, c = w.shape
            y = gpu.alloc_f32(batch * r)
            name, params = ("matvec_f16", [r, c]) if batch == 1 else ("matmul_f16", [r, c, batch])
            calls.append(_call(name, [_upload(w), _upload(x), y], params))
            out["y%d" % i] = (y, (batch, r))
        return {"calls": calls, "out": out, "logits": None}
    meta, fmt, suffix = case["meta"], [case["bits"], case["group"]], SUFFIX[case["meta"]]
    if kind == "mlp":
        for i, layer in enumerate(t["layers"]):
            x, h, y = _upload(layer["x"]), gpu.alloc_f32(batch * rows), gpu.alloc_f32(batch * cols)
            calls.append(_call("mlp_gate_up_swiglu" + suffix,
                               [*_upload_packed(layer["gate"], meta), *_upload_packed(layer["up"], meta), x,
                                _upload(layer["norm"]), h], [rows, cols, *fmt, batch, _eps_bits()]))
            calls.append(_call("matmul_affine_add" + suffix, [*_upload_packed(layer["down"], meta), h, x, y],
                               [cols, rows, *fmt, batch]))
            out["h%d" % i], out["y%d" % i] = (h, (batch, rows)), (y, (batch, cols))
        return {"calls": calls, "out": out, "logits": None}
    if kind == "embed":
        table, y = _upload_packed(t["matrices"][0], meta), gpu.alloc_f32(batch * cols)
        for i, token in enumerate(t["tokens"]):
            calls.append(_call("embed_affine" + suffix, [*table, y], [token, cols, *fmt], [0, 0, 0, 4 * i * cols]))
        return {"calls": calls, "out": {"x": (y, (batch, cols))}, "logits": None}
    xs = [_upload(x) for x in t["x"]]
    for i, (m, k) in enumerate(zip(t["matrices"], t["source"])):
        r, c = m[0].shape[0], t["x"][k].shape[1]
        y = gpu.alloc_f32(batch * r)
        if kind == "wide":
            name, params = "matmul_affine_wide" + suffix, [r, c, *fmt, batch]
        elif batch == 1:
            name, params = "matvec_affine" + suffix, [r, c, *fmt]
        else:
            name, params = "matmul_affine" + suffix, [r, c, *fmt, batch]
        calls.append(_call(name, [*_upload_packed(m, meta), xs[k], y], params))
        out["y%d" % i] = (y, (batch, r))
    return {"calls": calls, "out": out, "logits": out["y0"] if kind == "head" else None}


def run(state: dict):
    gpu = _gpu()
    command = gpu.begin()
    for name, buffers, params, threads, offsets in state["calls"]:
        command.encode(name, buffers, params, threads, 64, offsets)
    command.finish()
    command.release()
    if state["logits"] is not None:
        buffer, shape = state["logits"]
        return {"logits": gpu.read_f32(buffer, math.prod(shape)).reshape(shape)}
    return DeviceOutputs(state["out"])


# ---- what a pass cannot do without ----

def _shapes(case: dict) -> list[tuple[int, int]]:
    rows, cols = case["rows"], case["cols"]
    if case["kind"] == "dense":
        return [(rows, cols), (cols, rows)]
    if case["kind"] == "mlp" or case.get("shape") == "mlp":
        return [(rows, cols), (rows, cols), (cols, rows)] * case.get("layers", 1)
    return [(rows, cols)] * case.get("layers", 1)


def work(case: dict) -> dict:
    batch, cols = case["batch"], case["cols"]
    if case["kind"] == "embed":
        row = cols * case["bits"] / 8 + 2 * META_BYTES[case["meta"]] * cols / case["group"]
        return {"bytes": batch * (row + 4 * cols), "flops": 2.0 * batch * cols}
    per_weight = 2.0 if case["kind"] == "dense" else \
        case["bits"] / 8 + 2 * META_BYTES[case["meta"]] / case["group"]
    moved = flops = 0.0
    for r, c in _shapes(case):
        moved += per_weight * r * c + 4 * batch * (r + c)
        flops += 2.0 * batch * r * c
    return {"bytes": moved, "flops": flops}


# ---- correctness ----

def tolerance(case: dict):
    # Embedding rows are one FP32 rounding of scale * code + bias.
    if case["kind"] == "embed":
        return "exact"
    # FP32 sums over the columns: up to 8e-7 off the 64-bit result, and 2.2e-6
    # for the fused MLP, whose second launch carries on the first's rounding;
    # another order of the same sums may be four times that away.
    return {"rel": 9e-6 if case["kind"] == "mlp" else 3e-6}


def _dequantised(m, case: dict) -> torch.Tensor:
    """The packed matrix in 64 bits."""
    w, s, b = m
    bits, group = case["bits"], case["group"]
    shifts = torch.arange(0, 32, bits, device=w.device, dtype=torch.int32)
    q = ((w.unsqueeze(-1) >> shifts) & (2**bits - 1)).reshape(w.shape[0], -1, group).double()
    return (q * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).reshape(w.shape[0], -1)


def _product(x: torch.Tensor, m, case: dict) -> torch.Tensor:
    x = x.double()
    parts = []
    for i in range(0, m[0].shape[0], 16384):
        parts.append(x @ _dequantised([t[i:i + 16384] for t in m], case).T)
    return torch.cat(parts, dim=1)


def exact(case: dict, seed: int):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "dense":
        return {"y%d" % i: x.double() @ w.double().T for i, (w, x) in enumerate(zip(t["matrices"], t["x"]))}
    if kind == "embed":
        m = [v[t["tokens"]] for v in t["matrices"][0]]
        return {"x": _dequantised(m, case)}
    if kind == "mlp":
        out = {}
        eps = float(np.float32(EPS))
        for i, layer in enumerate(t["layers"]):
            x = layer["x"].double()
            n = x / torch.sqrt(x.square().mean(dim=1, keepdim=True) + eps) * layer["norm"].double()
            h = torch.nn.functional.silu(_product(n, layer["gate"], case)) * _product(n, layer["up"], case)
            out["h%d" % i], out["y%d" % i] = h, x + _product(h, layer["down"], case)
        return out
    y = [_product(t["x"][k], m, case) for m, k in zip(t["matrices"], t["source"])]
    return {"logits": y[0]} if kind == "head" else {"y%d" % i: v for i, v in enumerate(y)}
