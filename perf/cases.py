"""The calls whose time this framework is judged by: matrix products as inference programs make them, through the public
entry points (``vecops_amd.capi``, ``vecops_amd.torch_bridge``), from decode-shaped ones bound by launches and latency to
prefill-shaped ones bound by the matrix cores, with ragged extents and every operand class in earnest use.

``listed()`` names twelve of them, ``draw(rng)`` gives another of the same kinds and ranges, ``prepare`` makes what a
program holds before the call, ``run`` is one call.
"""
from __future__ import annotations

import math

import torch

from vecops_amd import capi, torch_bridge

# Matrix-core rate (operations a second) a call of this kind reaches at best: only to keep drawn cases below the largest
# listed one.
_RATES = {"bf16": 1.4e15, "f16": 1.4e15, "f32": 0.7e15, "f32c": 0.1e15, "i8": 2.2e15}
_TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "f32c": torch.float32, "i8": torch.int8}
_BYTES = {"bf16": 2, "f16": 2, "f32": 4, "f32c": 4, "i8": 1, "i32": 4}


def listed() -> list[dict]:
    return [
        # one token through a weight-only quantised projection: every byte of the weights is read once
        {"name": "weight_only_m1", "kind": "weight_only", "m": 1, "n": 14336, "k": 4096, "group": 128},
        # the same with sixteen sequences decoded together
        {"name": "weight_only_m16", "kind": "weight_only", "m": 16, "n": 14336, "k": 4096, "group": 128},
        # a decode step of a PyTorch program on unquantised weights, through the registered torch operator: the smallest
        # call, where what surrounds the kernel counts
        {"name": "torch_op_decode_m4", "kind": "torch_op", "dtype": "bf16", "m": 4, "n": 4096, "k": 4096, "out": "bf16"},
        # a short prompt's prefill: few rows, the weights' bytes weigh as much as the arithmetic
        {"name": "prefill_m128", "kind": "product", "dtype": "bf16", "m": 128, "n": 11008, "k": 4096, "layout": "nk",
         "out": "bf16", "cin": "none"},
        # the big square product, weights stored [K,N] as they are trained
        {"name": "square_4096", "kind": "prepared", "dtype": "bf16", "batch": 1, "m": 4096, "n": 4096, "k": 4096,
         "layout": "kn", "out": "bf16", "cin": "none"},
        # a batch of products with extents that line up with nothing
        {"name": "ragged_batch", "kind": "prepared", "dtype": "bf16", "batch": 8, "m": 777, "n": 1000, "k": 3001,
         "layout": "nk", "out": "f32", "cin": "none"},
        # a feed-forward layer of a long prompt: bias and silu in the product's epilogue (the largest case)
        {"name": "bias_silu", "kind": "fused", "dtype": "bf16", "m": 4096, "n": 11008, "k": 4096, "out": "bf16",
         "bias": True, "scales": False, "activation": "silu"},
        # an output projection added to the residual stream
        {"name": "residual_f16", "kind": "prepared", "dtype": "f16", "batch": 1, "m": 2048, "n": 4096, "k": 4096,
         "layout": "nk", "out": "f16", "cin": "full"},
        # int8 activations and weights, per-token and per-channel scales, dequantised fp32 results
        {"name": "int8_dequant", "kind": "int8_dequant", "m": 2048, "n": 11008, "k": 4096, "packed": False},
        # fp32 activations quantised on the way in against int8 weights packed once
        {"name": "runtime_quant", "kind": "runtime_quant", "m": 1000, "n": 4096, "k": 4096},
        # single-precision products that must keep single precision
        {"name": "fp32_1024", "kind": "prepared", "dtype": "f32c", "batch": 1, "m": 1024, "n": 1024, "k": 1024,
         "layout": "kn", "out": "f32", "cin": "none"},
        # unlike products in one call (experts with different token counts, irregular batches)
        {"name": "grouped", "kind": "grouped", "dtype": "bf16", "out": "bf16", "groups": 8, "tokens": 2048, "n": 4096,
         "k": 2048, "spread": 1},
    ]


def _size(rng, low: int, high: int, steps=(1, 1, 8, 64, 128)) -> int:
    """An extent between low and high, even over the logarithm; a good part of them multiples of what kernels like."""
    value = math.exp(rng.uniform(math.log(low), math.log(high)))
    step = rng.choice(steps)
    return int(min(high, max(low, round(value / step) * step)))


def _drawn(rng) -> dict:
    kind = rng.choice(["weight_only", "weight_only", "torch_op", "product", "product", "square", "batched", "fused",
                       "residual", "int8_dequant", "runtime_quant", "fp32", "grouped"])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    if kind == "weight_only":
        return {"kind": kind, "m": rng.randint(1, 16), "n": _size(rng, 1024, 16384), "k": _size(rng, 1024, 14336, (128,)),
                "group": rng.choice([64, 128, 128])}
    if kind == "torch_op":
        return {"kind": kind, "dtype": dtype, "m": rng.randint(1, 16), "n": _size(rng, 512, 16384),
                "k": _size(rng, 512, 14336, (1, 16, 64, 128)), "out": rng.choice([dtype, "f32"])}
    if kind == "product":
        dtype = rng.choice(["bf16", "bf16", "f16", "f32", "i8"])
        out = "i32" if dtype == "i8" else "f32" if dtype == "f32" else rng.choice([dtype, "f32"])
        return {"kind": kind, "dtype": dtype, "m": _size(rng, 17, 1024), "n": _size(rng, 256, 14336),
                "k": _size(rng, 256, 14336), "layout": "nk" if dtype == "i8" else rng.choice(["nk", "nk", "kn"]), "out": out,
                "cin": "none"}
    if kind == "square":
        return {"kind": "prepared", "dtype": dtype, "batch": 1, "m": _size(rng, 512, 8192), "n": _size(rng, 512, 8192),
                "k": _size(rng, 512, 8192), "layout": rng.choice(["nk", "kn"]), "out": rng.choice([dtype, "f32"]),
                "cin": "none"}
    if kind == "batched":
        return {"kind": "prepared", "dtype": dtype, "batch": rng.randint(2, 16), "m": _size(rng, 1, 3000),
                "n": _size(rng, 63, 4097), "k": _size(rng, 17, 8191), "layout": "nk", "out": "f32", "cin": "none"}
    if kind == "fused":
        return {"kind": kind, "dtype": dtype, "m": _size(rng, 17, 4096), "n": _size(rng, 256, 14336),
                "k": _size(rng, 256, 14336), "out": rng.choice([dtype, dtype, "f32"]), "bias": rng.random() < 0.7,
                "scales": rng.random() < 0.3, "activation": rng.choice(["none", "relu", "silu", "silu", "sigmoid"])}
    if kind == "residual":
        return {"kind": "prepared", "dtype": dtype, "batch": 1, "m": _size(rng, 17, 4096), "n": _size(rng, 256, 8192),
                "k": _size(rng, 256, 14336), "layout": rng.choice(["nk", "kn"]), "out": rng.choice([dtype, dtype, "f32"]),
                "cin": rng.choice(["full", "full", "bias"])}
    if kind == "int8_dequant":
        m = _size(rng, 1, 4096)
        return {"kind": kind, "m": m, "n": _size(rng, 512, 14336), "k": _size(rng, 512, 14336, (1, 16, 128)),
                "packed": m > 16 and rng.random() < 0.3}
    if kind == "runtime_quant":
        return {"kind": kind, "m": _size(rng, 17, 2048), "n": _size(rng, 512, 11008), "k": _size(rng, 512, 11008, (1, 16, 128))}
    if kind == "fp32":
        return {"kind": "prepared", "dtype": "f32c", "batch": 1, "m": _size(rng, 64, 2048), "n": _size(rng, 64, 2048),
                "k": _size(rng, 64, 4096), "layout": rng.choice(["nk", "kn"]), "out": "f32", "cin": "none"}
    return {"kind": kind, "dtype": dtype, "out": rng.choice([dtype, "f32"]), "groups": rng.randint(2, 24),
            "tokens": _size(rng, 64, 4096), "n": _size(rng, 256, 8192), "k": _size(rng, 256, 8192),
            "spread": rng.randint(1, 1000)}


def _cost(case: dict) -> float:
    w = work(case)
    dtype = "i8" if case["kind"] in ("int8_dequant", "runtime_quant") else case.get("dtype", "bf16")
    return max(w["bytes"] / 4e12, w["flops"] / _RATES[dtype])


def draw(rng) -> dict:
    """One more case of the listed kinds, at most two thirds of the largest listed one's cost."""
    most = max(_cost(c) for c in listed()) * 2 / 3
    while True:
        case = _drawn(rng)
        if _cost(case) <= most:
            return case


def _group_rows(case: dict) -> list[int]:
    """How many rows each product of a grouped call has: the tokens dealt unevenly, from one row on."""
    count, state, weights = case["groups"], case["spread"], []
    for _ in range(count):
        state = (state * 1103515245 + 12345) % (1 << 31)
        weights.append(0.15 + (state >> 8) / (1 << 23))
    total = sum(weights)
    return [max(1, round(case["tokens"] * w / total)) for w in weights]


class _Random:
    """Operands of one state, from its seed alone."""

    def __init__(self, seed: int):
        self.generator = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, shape, sigma, dtype):
        x = torch.randn(shape, generator=self.generator, device="cuda", dtype=torch.float32)
        return x.mul_(sigma).to(dtype)

    def bytes(self, shape):
        return torch.randint(-127, 128, shape, generator=self.generator, device="cuda", dtype=torch.int8)

    def scales(self, shape):
        return torch.rand(shape, generator=self.generator, device="cuda").add_(1.0).mul_(2.0 ** -7)


def _activations(r: _Random, case: dict, shape):
    return r.bytes(shape) if case["dtype"] == "i8" else r.normal(shape, 1.0, _TORCH[case["dtype"]])


def _weights(r: _Random, case: dict, batch, n: int, k: int):
    """b as the entry points take it, [..,N,K]: stored like that, or a view of weights stored [..,K,N]."""
    if case["dtype"] == "i8":
        return r.bytes((*batch, n, k))
    stored = (*batch, k, n) if case.get("layout") == "kn" else (*batch, n, k)
    w = r.normal(stored, 0.02, _TORCH[case["dtype"]])
    return w.transpose(-1, -2) if case.get("layout") == "kn" else w


def _out(case: dict, shape):
    kind = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "i32": torch.int32}[case["out"]]
    return torch.empty(shape, dtype=kind, device="cuda")


_ops = None


def _torch_operators():
    global _ops
    if _ops is None:
        _ops = torch_bridge.register_all()
    return _ops


def prepare(case: dict, seed: int):
    """Operands, outputs and what a program keeps from call to call; returns (the call, its arguments)."""
    r, kind = _Random(seed), case["kind"]
    if kind == "weight_only":
        m, n, k = case["m"], case["n"], case["k"]
        x, w = r.normal((m, k), 1.0, torch.bfloat16), r.bytes((n, k))
        return capi.matmul_w8a16_group, (x, w, r.scales((n, k // case["group"])),
                                         torch.empty((m, n), dtype=torch.bfloat16, device="cuda"), case["group"]), {}
    if kind == "torch_op":
        a, b = _activations(r, case, (case["m"], case["k"])), _weights(r, case, (), case["n"], case["k"])
        return _torch_operators().matmul, (a, b, None, _out(case, (case["m"], case["n"]))), {}
    compute = capi.COMPUTE_F32 if case.get("dtype") == "f32c" else capi.COMPUTE_BF16
    if kind in ("product", "prepared"):
        batch = (case["batch"],) if case.get("batch", 1) > 1 else ()
        a, b = _activations(r, case, (*batch, case["m"], case["k"])), _weights(r, case, batch, case["n"], case["k"])
        c, cin = _out(case, (*batch, case["m"], case["n"])), None
        if case["cin"] == "full":
            cin = r.normal((*batch, case["m"], case["n"]), 1.0, c.dtype)
        elif case["cin"] == "bias":
            cin = r.normal((case["n"],), 1.0, c.dtype).expand(*batch, case["m"], case["n"])
        if kind == "product":
            return capi.matmul, (a, b, c, cin, compute), {}
        return capi.PreparedMatmul(a, b, c, cin, compute), (), {}
    if kind == "fused":
        a, b = _activations(r, case, (case["m"], case["k"])), _weights(r, case, (), case["n"], case["k"])
        c = _out(case, (case["m"], case["n"]))
        bias = r.normal((case["n"],), 1.0, _TORCH[case["dtype"]]).expand(case["m"], case["n"]) if case["bias"] else None
        scales = r.scales((case["n"],)).mul_(64.0) if case["scales"] else None
        ep = capi.epilogue(activation=case["activation"], column_scales=scales)
        # (the descriptor holds the scales' address: they stay with the state)
        return _fused, (a, b, c, ep, bias, scales), {}
    if kind == "int8_dequant":
        m, n, k = case["m"], case["n"], case["k"]
        a, b, rows, columns = r.bytes((m, k)), r.bytes((n, k)), r.scales((m,)), r.scales((n,))
        c = torch.empty((m, n), dtype=torch.float32, device="cuda")
        if case["packed"]:
            return capi.matmul_i8_dequant_packed_b, (a, capi.pack_b(b), rows, columns, c), {}
        return capi.matmul_i8_dequant, (a, b, rows, columns, c), {}
    if kind == "runtime_quant":
        m, n, k, zero_point = case["m"], case["n"], case["k"], 128
        a = r.normal((m, k), 1.0, torch.float32)
        packed, correction = capi.pack_b(r.bytes((n, k)), a_zero_point=zero_point)
        multipliers = 127.0 / a.abs().amax(dim=1)
        c = torch.empty((m, n), dtype=torch.float32, device="cuda")
        return capi.matmul_runtime_quant_packed_b, (a, multipliers, zero_point, packed, 1.0 / multipliers, r.scales((n,)), c,
                                                    correction), {}
    a, b, c = [], [], []
    for rows in _group_rows(case):
        a.append(_activations(r, case, (rows, case["k"])))
        b.append(_weights(r, case, (), case["n"], case["k"]))
        c.append(_out(case, (rows, case["n"])))
    return capi.PreparedGrouped(a, b, c), (), {}


def _fused(a, b, c, ep, bias, scales):
    return capi.matmul_fused(a, b, c, ep, c_in=bias)


def run(state):
    call, arguments, named = state
    return call(*arguments, **named)


def work(case: dict) -> dict:
    kind, n, k = case["kind"], case["n"], case["k"]
    if kind == "grouped":
        rows, b, o = sum(_group_rows(case)), _BYTES[case["dtype"]], _BYTES[case["out"]]
        return {"bytes": rows * k * b + case["groups"] * n * k * b + rows * n * o, "flops": 2 * rows * n * k}
    batch, m = case.get("batch", 1), case["m"]
    flops = 2 * batch * m * n * k
    if kind == "weight_only":
        return {"bytes": 2 * m * k + n * k + 4 * n * (k // case["group"]) + 2 * m * n, "flops": flops}
    if kind == "int8_dequant":
        return {"bytes": m * k + n * k + 4 * m * n + 4 * (m + n), "flops": flops}
    if kind == "runtime_quant":
        return {"bytes": 4 * m * k + n * k + 4 * m * n + 8 * m + 8 * n, "flops": flops}
    b, o = _BYTES[case["dtype"]], _BYTES[case["out"]]
    more = batch * m * n * o if case.get("cin") == "full" else n * o if case.get("cin") == "bias" else 0
    if kind == "fused":
        more += (n * b if case["bias"] else 0) + (4 * n if case["scales"] else 0)
    return {"bytes": batch * (m * k + n * k) * b + batch * m * n * o + more, "flops": flops}


def tolerance(case: dict):
    # Integer sums and their dequantisation are exact by contract.
    if case["kind"] in ("int8_dequant", "runtime_quant") or case.get("dtype") == "i8":
        return "exact"
    # Against the same products in fp64, over these ranges: the rounding of a bf16 result is 1.7e-3 (largest 3.9e-3), of
    # an f16 one 2.1e-4 (4.9e-4), and fp32 sums of up to some ten thousand terms are off by up to 6e-7 (5e-6), which grows
    # with their number.  Four times that, and for fp32 a little more for another order of the sums.
    out = "bf16" if case["kind"] == "weight_only" else case["out"]
    return {"bf16": {"rel": 6.6e-3, "max": 1.6e-2}, "f16": {"rel": 8.4e-4, "max": 2e-3}, "f32": {"rel": 5e-6, "max": 5e-5}}[out]
