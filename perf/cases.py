"""Workloads of this library as a user's program runs them, for timing and for comparing two builds.

A program holds a Spec, device buffers and a stream, and enqueues the Spec again and again
(`Spec.run_async`); a program that keeps its tensors on the host calls `Spec.run_host`, the stand-in
for the emitted `kernel(...)`.  The listed cases go from the smallest call (a launch-bound Matmul of
320 outputs) to a terascale projection; `draw` gives further sizes, dtypes, layouts and options of the
same kinds of work.
"""
import math

import numpy as np
import torch

import morello_amd as M

_DTYPE = {"u8": M.u8, "i8": M.i8, "i32": M.i32, "f32": M.f32, "bf16": M.bf16}
_TORCH = {"u8": torch.uint8, "i8": torch.int8, "i32": torch.int32, "f32": torch.float32, "bf16": torch.bfloat16}
_NUMPY = {"u8": np.uint8, "i8": np.int8, "i32": np.int32, "f32": np.float32}
_SIZE = {"u8": 1, "i8": 1, "i32": 4, "f32": 4, "bf16": 2}
# Operand and result dtypes of a Matmul or Conv by their short name.
_TYPES = {
    "u8i8": ("u8", "i8", "i32"),          # quantised: the result is exact
    "bf16": ("bf16", "bf16", "f32"),      # bf16 operands, the sums as they were formed
    "bf16_out": ("bf16", "bf16", "bf16"),  # bf16 throughout, as one layer hands to the next
    "f32": ("f32", "f32", "f32"),
}


def _matmul(types, m, k, n, b=1, weights="kn", accum=False, host=False):
    return {"op": "matmul", "types": types, "b": b, "m": m, "k": k, "n": n, "weights": weights, "accum": accum, "host": host}


def _conv(types, b, c, f, oh, ow, fh, fw):
    return {"op": "conv", "types": types, "b": b, "c": c, "f": f, "oh": oh, "ow": ow, "fh": fh, "fw": fw}


def _softmax(b, rows, cols, dim, host=False):
    return {"op": "softmax", "b": b, "rows": rows, "cols": cols, "dim": dim, "host": host}


def _attention(types, b, m, keys, d, host=False):
    return {"op": "attention", "types": types, "b": b, "m": m, "keys": keys, "d": d, "host": host}


def _move(source, dest, rows, cols, into):
    return {"op": "move", "from": source, "to": dest, "rows": rows, "cols": cols, "into": into}


def listed():
    return [
        # The smallest call a program makes: a classifier's last layer, all latency and launch.
        dict(_matmul("f32", 32, 256, 10), name="matmul_f32_head"),
        # The headline workload: quantised Matmul accumulating into its output.
        dict(_matmul("u8i8", 4096, 4096, 4096, accum=True), name="matmul_u8i8_4096_accum"),
        # A long prompt through a large projection whose weights are stored output-major, as checkpoints hold them.
        dict(_matmul("bf16", 8192, 8192, 8192, weights="nk"), name="linear_bf16_8192"),
        # A prompt of an odd number of tokens through layers of odd widths, bf16 in and out.
        dict(_matmul("bf16_out", 1001, 2050, 4425), name="matmul_bf16_ragged"),
        # Decoding one token: a matrix-vector product, a stream over the weights.
        dict(_matmul("bf16", 1, 2048, 16384, weights="nk"), name="linear_bf16_decode"),
        # A body layer of a quantised convolutional network.
        dict(_conv("u8i8", 32, 64, 64, 54, 54, 3, 3), name="conv_u8i8_body"),
        # Its bf16 first layer: three channels, wide filters, an odd image.
        dict(_conv("bf16", 16, 3, 64, 109, 109, 7, 7), name="conv_bf16_first"),
        # Normalising attention scores of a sequence of odd length.
        dict(_softmax(16, 1501, 1501, 2), name="softmax_f32_odd"),
        # Attention over a prompt (prefill).
        dict(_attention("bf16", 16, 2048, 2048, 128), name="attention_prefill"),
        # Attention of one new token per sequence over a long cache (decode).
        dict(_attention("bf16", 16, 1, 32768, 128), name="attention_decode"),
        # Packing a weight matrix into column strips before it is used: conversion and re-layout in one pass.
        dict(_move("f32", "bf16", 2048, 16384, "strips16"), name="move_pack_weights"),
        # The f32 Matmul -> Softmax -> Matmul chain called on host buffers, as an emitted program's main calls it.
        dict(_attention("f32", 1, 2048, 2048, 2048, host=True), name="chain_f32_host"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _side(rng, lo, hi):
    """A size: half of them round (whole tiles of 64), half as they come."""
    v = _log(rng, lo, hi)
    return max(64, v // 64 * 64) if rng.random() < 0.5 and v >= 64 else v


def draw(rng):
    kind = rng.randrange(12)
    if kind == 0:  # small Matmuls
        return _matmul(rng.choice(["f32", "bf16", "u8i8"]), _log(rng, 8, 256), _log(rng, 64, 512), _log(rng, 8, 256),
                       accum=rng.random() < 0.5)
    if kind == 1:  # large quantised ones
        return _matmul("u8i8", _side(rng, 1024, 6000), _side(rng, 1024, 6000), _side(rng, 1024, 6000),
                       weights=rng.choice(["kn", "nk"]), accum=rng.random() < 0.5)
    if kind == 2:  # large projections
        return _matmul(rng.choice(["bf16", "bf16_out"]), _side(rng, 1024, 8192), _side(rng, 1024, 8192), _side(rng, 1024, 8192),
                       weights=rng.choice(["kn", "nk"]), accum=rng.random() < 0.25)
    if kind == 3:  # middling, any size, several of them at once now and then
        return _matmul(rng.choice(["bf16", "bf16_out", "u8i8", "f32"]), _log(rng, 128, 2500), _log(rng, 128, 2500),
                       _log(rng, 128, 4500), b=rng.choice([1, 1, 1, 2]), weights=rng.choice(["kn", "nk"]))
    if kind == 4:  # decoding some tokens
        return _matmul(rng.choice(["bf16", "bf16", "u8i8"]), _log(rng, 1, 64), _side(rng, 1024, 12288), _side(rng, 1024, 16384), weights="nk")
    if kind == 5:  # body layers
        c, f, fs, hw = 16 * _log(rng, 1, 24), 16 * _log(rng, 1, 24), rng.choice([1, 3, 3, 5]), _log(rng, 7, 80)
        most = max(1, int(2e11 / (2 * c * f * fs * fs * hw * hw)))  # images; the wide and large layers run few at a time
        return _conv(rng.choice(["u8i8", "bf16"]), min(most, _log(rng, 1, 32)), c, f, hw, hw, fs, fs)
    if kind == 6:  # first layers
        hw, fs = _log(rng, 48, 224), rng.choice([3, 5, 7])
        return _conv(rng.choice(["u8i8", "bf16"]), _log(rng, 1, 32), rng.choice([3, 3, 4]), rng.choice([16, 32, 64, 96]), hw, hw, fs, fs)
    if kind == 7:  # Softmax along the rows, or along an outer dim
        return _softmax(_log(rng, 1, 32), _log(rng, 8, 2048), _side(rng, 16, 4096), rng.choice([2, 2, 2, 1]))
    if kind == 8:  # prefill
        return _attention("bf16", _log(rng, 1, 48), _side(rng, 64, 2048), _side(rng, 64, 2048), rng.choice([32, 64, 80, 96, 128, 128]))
    if kind == 9:  # decode
        return _attention("bf16", _log(rng, 1, 128), rng.choice([1, 1, 1, 2, 4, 8]), _side(rng, 256, 12288), rng.choice([64, 128]))
    if kind == 10:  # re-layouts: transposes, packed strips, even and odd elements apart, conversions
        source, dest = rng.choice([("f32", "bf16"), ("f32", "f32"), ("bf16", "bf16"), ("u8", "u8"), ("bf16", "f32"), ("u8", "f32")])
        return _move(source, dest, 16 * _log(rng, 4, 512), 16 * _log(rng, 4, 512), rng.choice(["turned", "strips16", "strips8", "rows16", "oddeven16"]))
    what = rng.randrange(3)  # on host buffers
    if what == 0:
        return _matmul(rng.choice(["f32", "u8i8"]), _log(rng, 32, 2048), _log(rng, 32, 2048), _log(rng, 32, 2048), host=True)
    if what == 1:
        return _softmax(1, _log(rng, 32, 2048), _log(rng, 32, 2048), 2, host=True)
    return _attention("f32", 1, _log(rng, 64, 2048), _log(rng, 64, 2048), _log(rng, 64, 2048), host=True)


# How a Move's destination stores a [1, rows, cols] tensor.
_INTO = {
    "turned": lambda: M.layout(0, 2, 1),                        # column-major
    "strips16": lambda: M.layout(0, 2, 1, (2, M.Packed(16))),   # strips of 16 columns: the right operand of a tiled Matmul
    "strips8": lambda: M.layout(0, 2, 1, (2, M.Packed(8))),
    "rows16": lambda: M.layout(0, 1, 2, (1, M.Packed(16))),     # strips of 16 rows: its left operand
    "oddeven16": lambda: M.layout(0, 1, 2, (2, M.OddEven(16))),  # even and odd elements of 16 apart, for widening bf16 in pairs
}

_stream = None


def _the_stream():
    """The program's stream: one for everything it enqueues."""
    global _stream
    if _stream is None:
        M.init(0)
        _stream = M.Stream()
    return _stream


def _device_tensor(gen, dtype, shape, std):
    if dtype in ("u8", "i8"):
        lo = 0 if dtype == "u8" else -128
        return torch.randint(lo, lo + 256, shape, generator=gen, device="cuda", dtype=_TORCH[dtype])
    return (torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * std).to(_TORCH[dtype])


def _host_tensor(gen, dtype, shape, std):
    if dtype in ("u8", "i8"):
        info = np.iinfo(_NUMPY[dtype])
        return gen.integers(info.min, info.max + 1, shape, dtype=_NUMPY[dtype])
    return gen.standard_normal(shape, dtype=np.float32) * np.float32(std)


def _spec(case):
    """The Spec of a case, its parameters as (dtype, stored shape), and the inputs' standard deviation."""
    op = case["op"]
    if op == "matmul":
        types = _TYPES[case["types"]]
        b, m, k, n = case["b"], case["m"], case["k"], case["n"]
        nk = case["weights"] == "nk"
        spec = M.Matmul([b, m, k, n], [_DTYPE[t] for t in types], [None, M.layout(0, 2, 1) if nk else None, None], case["accum"])
        shapes = [(b, m, k), (b, n, k) if nk else (b, k, n), (b, m, n)]
        return spec, list(zip(types, shapes)), 0.5
    if op == "conv":
        types = _TYPES[case["types"]]
        b, c, f, oh, ow, fh, fw = (case[x] for x in ("b", "c", "f", "oh", "ow", "fh", "fw"))
        spec = M.Conv([b, f, c, oh, ow, fh, fw], [_DTYPE[t] for t in types])
        shapes = [(b, oh + fh - 1, ow + fw - 1, c), (f, fh, fw, c), (b, oh, ow, f)]
        return spec, list(zip(types, shapes)), 0.5
    if op == "softmax":
        shape = (case["b"], case["rows"], case["cols"])
        return M.Softmax(list(shape), case["dim"]), [("f32", shape)] * 2, 2.0
    if op == "attention":
        b, m, keys, d, t = case["b"], case["m"], case["keys"], case["d"], case["types"]
        # bf16: K as the cache stores it, a row per key; f32: the reference chain's row-major operands.
        layouts = [None, None, M.layout(0, 2, 1), None] if t == "bf16" else None
        spec = M.ComposeMSM(b, m, d, keys, d, [_DTYPE[t]] * 3 + [M.f32], layouts)
        shapes = [(b, keys, d), (b, m, d), (b, keys, d) if t == "bf16" else (b, d, keys), (b, m, d)]
        # scores of a standard deviation of about 2
        return spec, list(zip([t, t, t, "f32"], shapes)), math.sqrt(2.0 / math.sqrt(d))
    shape = (1, case["rows"], case["cols"])
    spec = M.Move(list(shape), [_DTYPE[case["from"]], _DTYPE[case["to"]]], [None, _INTO[case["into"]]()])
    return spec, [(case["from"], shape), (case["to"], (case["rows"] * case["cols"],))], 1.0


def prepare(case, seed):
    spec, params, std = _spec(case)
    if case.get("host"):
        gen = np.random.default_rng(seed)
        tensors = [_host_tensor(gen, dtype, shape, std) for dtype, shape in params[:-1]]
        dtype, shape = params[-1]
        tensors.append(np.zeros(shape, _NUMPY[dtype]))
        M.init(0)
        return {"spec": spec, "tensors": tensors, "stream": None}
    gen = torch.Generator(device="cuda").manual_seed(seed)
    tensors = [_device_tensor(gen, dtype, shape, std) for dtype, shape in params[:-1]]
    dtype, shape = params[-1]
    tensors.append(torch.zeros(shape, dtype=_TORCH[dtype], device="cuda"))
    return {"spec": spec, "tensors": tensors, "ptrs": [t.data_ptr() for t in tensors], "stream": _the_stream()}


def run(state):
    if state["stream"] is None:
        state["spec"].run_host(*state["tensors"])
    else:
        state["spec"].run_async(state["ptrs"], state["stream"])
    return state["tensors"][-1]


def work(case):
    spec, params, _ = _spec(case)
    nbytes = sum(_SIZE[dtype] * math.prod(shape) for dtype, shape in params)
    if case.get("accum"):  # the old output is an input
        nbytes += _SIZE[params[-1][0]] * math.prod(params[-1][1])
    return {"bytes": nbytes, "flops": 0 if case["op"] == "move" else spec.flops()}


def tolerance(case):
    op, types = case["op"], case.get("types")
    if op == "move" or types == "u8i8":
        return "exact"
    if op == "softmax":
        return {"rel": 1e-5}
    if op == "attention":
        # bf16: the probabilities are rounded to bf16 before the second product
        return {"rel": 5e-3} if types == "bf16" else {"rel": 2e-5}
    if types == "bf16_out":
        # f32 sums rounded once: a sum near a tie may fall to the neighbouring bf16
        return {"rel": 2e-3, "max": 1.6e-2}
    return {"rel": 1e-5}
