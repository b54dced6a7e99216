"""The work this library is used for, as cases that can be timed.

A decode step of a language model with int4 or int8 weights is a chain of matrix-vector products: a few
activation rows against every projection of every layer, then against the vocabulary.  The cases are such
calls from the smallest (a key/value projection, where the call itself costs more than the product) to the
largest (a vocabulary projection), the expert products of a mixture layer, a whole stretch of decoder layers,
and the two things done beside decoding: weights brought into the library's layout when a model is loaded,
and matrices expanded to 16 bits for a prefill's dense product.  Shapes and value distributions are those of
the benchmark's workloads and the tests; the rest are generic.

kind     what one pass is
gemv     one product, m activation rows
layers   the projections of `layers` decoder layers: q/k/v in one batched launch, o, gate/up in one batched
         launch, down
routed   the products of one token with `top` of `experts` matrices, chosen by indices on the device
expand   one matrix dequantised to 16 bits
load     one matrix as a checkpoint holds it (one int4 per byte, integer zero points) packed, laid out, and its
         zero points folded, on the host
"""
import math

import numpy as np
import torch

import mixed_gemv_amd as mg

PER_COLUMN, SCALE_ONLY, SCALE_ZERO = 1, 2, 3


def _case(kind, n_out, k, bits=4, op=SCALE_ZERO, group=128, m=1, bias=False, element="f16", name=None, **more):
    case = {"kind": kind, "n_out": n_out, "k": k, "bits": bits, "op": op, "group": group, "m": m, "bias": bias,
            "element": element, **more}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # the smallest call of a decode step: a grouped key or value projection
        _case("gemv", 1024, 2048, name="kv_projection"),
        # the benchmark's headline: a square attention projection, one token
        _case("gemv", 4096, 4096, name="attention_projection"),
        # int8 weights with one scale per column, as 8-bit exporters write them
        _case("gemv", 4096, 4096, bits=8, op=PER_COLUMN, bias=True, name="int8_projection"),
        # sizes that fit no tile: odd row count, a group that is no power of two, a few speculative tokens
        _case("gemv", 5004, 5280, op=SCALE_ONLY, group=96, m=3, bias=True, element="bf16", name="ragged_bf16"),
        # several requests decoded together on a square projection with fine groups
        _case("gemv", 8192, 8192, group=64, m=16, bias=True, name="projection_batch16"),
        # a large model's up projection, one token
        _case("gemv", 28672, 8192, name="mlp_up"),
        # the same matrix where the model runs in bfloat16
        _case("gemv", 28672, 8192, element="bf16", name="mlp_up_bf16"),
        # the vocabulary projection, the longest product of a decode step, a small batch in bfloat16
        _case("gemv", 128256, 4096, m=4, element="bf16", name="vocabulary_bf16"),
        # one token through a mixture layer: 8 of 64 experts in one launch
        _case("routed", 1408, 2048, experts=64, top=8, name="experts"),
        # one token through four decoder layers, weights coming from memory as in a real step
        _case("layers", 4096, 11008, layers=4, name="decoder_layers"),
        # a matrix expanded for the dense product of a prefill
        _case("expand", 11008, 4096, name="expand"),
        # one matrix of a checkpoint being loaded
        _case("load", 4096, 4096, name="load"),
    ]


def _log(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _multiple(value, of):
    return max(of, int(round(value / of)) * of)


def draw(rng):
    kind = rng.choice(["gemv"] * 7 + ["routed", "layers", "expand", "load"])
    bits = 4 if kind == "load" else rng.choice([4, 4, 4, 8])
    op = SCALE_ZERO if kind == "load" else rng.choice([SCALE_ZERO, SCALE_ZERO, SCALE_ONLY, PER_COLUMN])
    group = rng.choice([64, 128, 128, 128, 96, 256])
    element = "f16" if kind == "load" else rng.choice(["f16", "f16", "bf16"])
    bias = kind == "gemv" and rng.random() < 0.4
    step = 8 if op == PER_COLUMN else group  # k is whole groups
    if kind == "gemv":
        most = 128256 * 4096 // 2
        k = _multiple(_log(rng, 1024, 28672), step)
        n_out = _multiple(_log(rng, 512, min(152064, most * 8 // bits / k)), 4)
        m = rng.choice([1, 1, 1, 1, 2, 3, 4, 6, 8, 12, 16])
        return _case(kind, n_out, k, bits, op, group, m, bias, element)
    if kind == "routed":
        experts = rng.choice([8, 16, 32])
        k = _multiple(_log(rng, 1024, 2816), step)
        n_out = _multiple(_log(rng, 768, 2816), 4)
        return _case(kind, n_out, k, bits, op, group, 1, False, element, experts=experts, top=rng.randint(2, 8))
    if kind == "layers":
        hidden = _multiple(_log(rng, 1024, 4096), step)
        inner = _multiple(hidden * rng.uniform(2.0, 2.68), step)
        return _case(kind, hidden, inner, bits, op, group, rng.choice([1, 1, 2, 4]), False, element, layers=2)
    n_out = _multiple(_log(rng, 512, 11008 if kind == "expand" else 4096), 4)
    k = _multiple(_log(rng, 512, 4096), step)
    return _case(kind, n_out, k, bits, op, group, 1, False, element)


def _quant_type(case):
    return mg.QuantType.W4_A16 if case["bits"] == 4 else mg.QuantType.W8_A16


def _dtype(case):
    return torch.bfloat16 if case["element"] == "bf16" else torch.half


def _groups(case, k):
    return 1 if case["op"] == PER_COLUMN else k // case["group"]


class _Matrices:
    """`count` matrices of one shape, stacked: laid out weights, scales, folded zeros, on the GPU."""

    def __init__(self, case, gen, n_out, k, count=1):
        dt, dev = _dtype(case), "cuda"
        raw = torch.randint(0, 256, (count * n_out * k * case["bits"] // 8,), dtype=torch.uint8, device=dev, generator=gen)
        laid_out = mg.MixedGemvWeightPreprocessor.run(raw.cpu().numpy(), (count, k, n_out), mg.LayoutType.kColumnMajor,
                                                      _quant_type(case))
        self.w = torch.from_numpy(laid_out).to(dev)
        table = (count, _groups(case, k), n_out)
        # 8-bit scales are smaller than 4-bit ones, as the integers are larger
        low, high = (0.001, 0.02) if case["bits"] == 4 else (0.0005, 0.01)
        self.s = (torch.rand(table, device=dev, generator=gen) * (high - low) + low).to(dt)
        self.z = (torch.rand(table, device=dev, generator=gen) * 0.1 - 0.05).to(dt) if case["op"] == SCALE_ZERO else None
        self.n_out, self.k, self.count = n_out, k, count
        # strides of a batched or routed launch: weights in bytes, x (shared), scales, bias, y in elements
        self.strides = (self.w.numel() // count, 0, table[1] * n_out, 0, case["m"] * n_out)


def _activations(case, gen, k):
    return torch.randn((case["m"], k), device="cuda", generator=gen).clamp_(-4, 4).to(_dtype(case))


def _outputs(case, n_out, count=1):
    return torch.zeros((count, case["m"], n_out), dtype=_dtype(case), device="cuda")


def prepare(case, seed):
    kind, n_out, k = case["kind"], case["n_out"], case["k"]
    state = {"case": case}
    if kind == "load":
        rng = np.random.default_rng(seed)
        state["q"] = rng.integers(-8, 8, (n_out, k), dtype=np.int8)
        state["s"] = (rng.random((_groups(case, k), n_out), dtype=np.float32) * 0.019 + 0.001).astype(np.float16)
        state["zeros"] = rng.integers(-8, 8, state["s"].shape, dtype=np.int8)
        return state
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if kind == "gemv":
        state["mat"] = _Matrices(case, gen, n_out, k)
        state["x"] = _activations(case, gen, k)
        state["bias"] = (torch.rand((n_out,), device="cuda", generator=gen) * 0.2 - 0.1).to(_dtype(case)) if case["bias"] else None
        state["y"] = _outputs(case, n_out)
    elif kind == "routed":
        state["mat"] = _Matrices(case, gen, n_out, k, case["experts"])
        state["x"] = _activations(case, gen, k)
        state["route"] = torch.randperm(case["experts"], device="cuda", generator=gen)[:case["top"]].to(torch.int32)
        state["y"] = _outputs(case, n_out, case["top"])
    elif kind == "layers":
        hidden, inner = n_out, k
        state["calls"] = []
        for _ in range(case["layers"]):
            for rows, cols, count in ((hidden, hidden, 3), (hidden, hidden, 1), (inner, hidden, 2), (hidden, inner, 1)):
                mat = _Matrices(case, gen, rows, cols, count)
                state["calls"].append((mat, _activations(case, gen, cols), _outputs(case, rows, count)))
    elif kind == "expand":
        state["mat"] = _Matrices(case, gen, n_out, k)
        state["out"] = torch.empty((n_out, k), dtype=_dtype(case), device="cuda")
    return state


def run(state):
    case = state["case"]
    kind, op, bits, group, m = case["kind"], case["op"], case["bits"], case["group"], case["m"]
    if kind == "gemv":
        mat = state["mat"]
        mg.device_gemv(mat.w, state["x"], mat.s, mat.z, state["bias"], state["y"], 1, mat.n_out, m, mat.k, group, op, bits)
        return state["y"]
    if kind == "routed":
        mat = state["mat"]
        mg.device_gemv_routed(mat.w, state["x"], mat.s, mat.z, None, state["y"], state["route"], mat.count, case["top"],
                              mat.n_out, m, mat.k, group, mat.strides, op, bits)
        return state["y"]
    if kind == "layers":
        for mat, x, y in state["calls"]:
            mg.device_gemv(mat.w, x, mat.s, mat.z, None, y, mat.count, mat.n_out, m, mat.k, group, op, bits,
                           batch_strides=mat.strides if mat.count > 1 else None)
        return [y for _, _, y in state["calls"]]
    if kind == "expand":
        mat = state["mat"]
        mg.dequantize(mat.w, mat.s, mat.z, state["out"], mat.n_out, mat.k, group, op, bits)
        return state["out"]
    packed = mg.SubBytePacker.pack(state["q"])
    weights = mg.MixedGemvWeightPreprocessor.run(packed, (case["k"], case["n_out"]), mg.LayoutType.kColumnMajor, _quant_type(case))
    zero_add = mg.ZeroPointPreprocessor.neg_zero_point_multiplies_scale(state["s"], state["zeros"])
    return weights, zero_add


def work(case):
    kind, n_out, k, m = case["kind"], case["n_out"], case["k"], case["m"]

    def matrix(rows, cols):
        return rows * cols * case["bits"] // 8 + _groups(case, cols) * rows * 2 * (2 if case["op"] == SCALE_ZERO else 1)

    if kind == "gemv":
        return {"bytes": matrix(n_out, k) + (n_out * 2 if case["bias"] else 0) + m * k * 2 + m * n_out * 2,
                "flops": 2 * m * n_out * k}
    if kind == "routed":
        return {"bytes": case["top"] * (matrix(n_out, k) + m * n_out * 2 + 4) + m * k * 2,
                "flops": 2 * case["top"] * m * n_out * k}
    if kind == "layers":
        total, flops = 0, 0
        for rows, cols, count in ((n_out, n_out, 3), (n_out, n_out, 1), (k, n_out, 2), (n_out, k, 1)):
            total += count * (matrix(rows, cols) + m * rows * 2) + m * cols * 2
            flops += 2 * count * m * rows * cols
        return {"bytes": case["layers"] * total, "flops": case["layers"] * flops}
    if kind == "expand":
        return {"bytes": matrix(n_out, k) + n_out * k * 2, "flops": 2 * n_out * k}
    # one byte per integer in, half a byte out; a scale and an integer zero in, a folded zero out
    return {"bytes": n_out * k * 3 // 2 + _groups(case, k) * n_out * 5, "flops": 0}


def tolerance(case):
    if case["kind"] in ("expand", "load"):
        return "exact"
    # the outputs' own rounding, and 32-bit sums in another order in front of it
    return {"rel": 8e-3, "max": 4e-2} if case["element"] == "bf16" else {"rel": 1e-3, "max": 5e-3}
