"""The work a caller of this library has it do, as timed cases.

Every case builds one KernelModule with mlkhip_build and runs it on device
buffers with mlkhip_run_device, as a caller of include/mlk_hip.h does: the
artifact and the binding array are made once, each pass is one call on the
default stream. The device buffers are torch tensors, so inputs are drawn on
the GPU and outputs come back without a copy.

A case is a dict: "kind" (softmax, chain, broadcast, gemm, score), its sizes
and its options. `listed` holds the named ones; `draw` gives others of the
same ranges.
"""
from __future__ import annotations

import ctypes
import math

import torch

from mlk2_amd import fixtures as fx
from mlk2_amd.backend import DTYPE_CODE, Binding, last_error, lib
from mlk2_amd.kernel_ir import KernelExpr, KernelModule, const, elem_a, temp

TORCH = {"f16": torch.float16, "f32": torch.float32, "f64": torch.float64}
BYTES = {"f16": 2, "f32": 4, "f64": 8}


def listed():
    return [
        # A class head over one small batch: the call is latency and launches.
        dict(name="softmax_64x64", kind="softmax", rows=64, cols=64, dtype="f32"),
        # The headline: attention-sized rows over a large batch.
        dict(name="softmax_8192x4096", kind="softmax", rows=8192, cols=4096, dtype="f32"),
        # A vocabulary-sized output layer, its row length odd.
        dict(name="softmax_1000x30001", kind="softmax", rows=1000, cols=30001, dtype="f32"),
        # A fused elementwise chain over a large flat tensor.
        dict(name="chain_sin_16m", kind="chain", n=1 << 24, dtype="f32", op="sin"),
        # A chain with a row-broadcast operand (an activation with a bias).
        dict(name="broadcast_4096x4096", kind="broadcast", rows=4096, cols=4096, dtype="f32"),
        # Single-precision and double-precision products of ordinary size;
        # double is the type the reference itself computes in.
        dict(name="gemm_f32_1024", kind="gemm", m=1024, k=1024, n=1024, dtype="f32", call=False),
        dict(name="gemm_f64_512", kind="gemm", m=512, k=512, n=512, dtype="f64", call=False),
        # The large half-precision product.
        dict(name="gemm_f16_4096", kind="gemm", m=4096, k=4096, n=4096, dtype="f16", call=False),
        # C += A B at sizes off every tile.
        dict(name="gemm_f16_call_2000x1000x3000", kind="gemm", m=2000, k=1000, n=3000, dtype="f16", call=True),
        # A layer applied to a few rows (one decode step of a small batch).
        dict(name="gemm_f16_16x4096x4096", kind="gemm", m=16, k=4096, n=4096, dtype="f16", call=False),
        # Attention probabilities, long sequences and head dim 128, then a
        # smaller problem with head dim 64.
        dict(name="score_16x2048x128", kind="score", batch=16, seq=2048, dim=128),
        dict(name="score_8x1024x64", kind="score", batch=8, seq=1024, dim=64),
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], uniform over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["softmax", "softmax", "chain", "broadcast", "gemm", "gemm", "gemm", "score"])
    if kind == "softmax":
        cols = _log(rng, 8, 65536)
        rows = _log(rng, 1, max(1, min(16384, (1 << 25) // cols)))
        return dict(kind=kind, rows=rows, cols=cols, dtype=rng.choice(["f32", "f32", "f32", "f16"]))
    if kind == "chain":
        dtype = rng.choice(["f32", "f32", "f16", "f64"])
        return dict(kind=kind, n=_log(rng, 1 << 10, 1 << (23 if dtype == "f64" else 24)), dtype=dtype,
                    op=rng.choice(["sin", "exp"]))
    if kind == "broadcast":
        cols = _log(rng, 16, 16384)
        return dict(kind=kind, rows=_log(rng, 1, (1 << 24) // cols), cols=cols, dtype=rng.choice(["f32", "f32", "f16"]))
    if kind == "gemm":
        dtype = rng.choice(["f16", "f16", "f32", "f64"])
        most = {"f16": 1 << 37, "f32": 1 << 33, "f64": 1 << 28}[dtype]
        while True:
            k, n = _log(rng, 32, 8192), _log(rng, 32, 8192)
            m = _log(rng, 1, 64) if rng.random() < 0.35 else _log(rng, 32, 4096)
            if 2 * m * k * n <= most and m * k + k * n <= 1 << 26:
                return dict(kind=kind, m=m, k=k, n=n, dtype=dtype, call=rng.random() < 0.5)
    batch = _log(rng, 1, 16)
    if rng.random() < 0.4:
        return dict(kind=kind, batch=batch, seq=128 * rng.randint(1, 16), dim=64)
    return dict(kind=kind, batch=batch, seq=_log(rng, 64, 2048), dim=128)


def _module(c) -> KernelModule:
    kind = c["kind"]
    if kind == "softmax":
        return fx.softmax_call_module(c["rows"], c["cols"], c["dtype"])
    if kind == "chain":
        if c["op"] == "sin":
            return fx.config1_module(n=c["n"], dtype=c["dtype"])
        # y = exp(-x^2 / 2) * x
        chain = [KernelExpr("mul", elem_a(), elem_a()), KernelExpr("mul", const(-0.5), temp(0)),
                 KernelExpr("exp", temp(1), const(0.0)), KernelExpr("mul", temp(2), elem_a())]
        return fx.lower_elementwise([("x", [c["n"]], c["dtype"])], chain, [c["n"]], c["dtype"])
    if kind == "broadcast":
        return fx.synth_elementwise(fx.config3_tier1_module(c["rows"], c["cols"], c["dtype"]))
    if kind == "gemm":
        call = fx.matmul_call_module(c["m"], c["k"], c["n"], c["dtype"], "f64" if c["dtype"] == "f64" else "f32")
        return call if c["call"] else fx.synth_gemm(call)
    return fx.score_softmax_module(c["batch"], c["seq"], c["dim"])


def _inputs(c, seed):
    """(inputs in buffer order, output shape, output dtype, the output's first
    contents or None for zeros)."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFFFFFF)

    def uniform(shape, lo, hi, dtype):
        return (torch.rand(shape, generator=g, device="cuda", dtype=torch.float32) * (hi - lo) + lo).to(TORCH[dtype])

    def normal(shape, std, dtype):
        return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std).to(TORCH[dtype])

    kind = c["kind"]
    if kind == "softmax":
        shape = (c["rows"], c["cols"])
        return [normal(shape, 2.0, c["dtype"])], shape, c["dtype"], None
    if kind == "chain":
        return [uniform((c["n"],), -4.0, 4.0, c["dtype"])], (c["n"],), c["dtype"], None
    if kind == "broadcast":
        shape = (c["rows"], c["cols"])
        return ([uniform(shape, -2.0, 2.0, c["dtype"]), uniform((c["cols"],), -1.0, 1.0, c["dtype"])], shape,
                "f32", None)
    if kind == "gemm":
        m, k, n, out = c["m"], c["k"], c["n"], "f64" if c["dtype"] == "f64" else "f32"
        ins = [uniform((m, k), -1.0, 1.0, c["dtype"]), uniform((k, n), -1.0, 1.0, c["dtype"])]
        return ins, (m, n), out, uniform((m, n), -1.0, 1.0, out) if c["call"] else None
    b, s, d = c["batch"], c["seq"], c["dim"]
    return ([normal((b, s, d), 1.0, "f16"), normal((b, s, d), 1.0, "f16"), normal((s,), 0.1, "f32")], (b * s, s),
            "f32", None)


class _State:
    """A built artifact with its device buffers and binding array."""

    def __init__(self, c, seed):
        L = lib()
        km = _module(c)
        doc = km.to_json().encode()
        self.handle = ctypes.c_void_p()
        if L.mlkhip_build(doc, len(doc), b"gfx950", b"", ctypes.byref(self.handle)) != 0:
            raise RuntimeError(last_error())
        ins, shape, dtype, first = _inputs(c, seed)
        self.out = torch.zeros(shape, device="cuda", dtype=TORCH[dtype]) if first is None else first
        self.ins = ins
        ids = km.bindable_ids()
        bound = iter(ins)
        self.binds = (Binding * len(ids))()
        for i, bid in enumerate(ids):
            b = km.buffers[bid]
            if b.is_temp:
                self.binds[i] = Binding(None, 0, DTYPE_CODE[b.dtype], 0)
                continue
            t = next(bound) if b.is_input else self.out
            self.binds[i] = Binding(t.data_ptr(), t.numel(), DTYPE_CODE[b.dtype], 0)
        self.scalars = (ctypes.c_double * 1)(0.0)
        self.elements = c["n"] if c["kind"] == "chain" else 0
        self.call = L.mlkhip_run_device
        self.args = (self.handle, self.binds, len(ids), self.scalars, 0, self.elements, None)

    def __del__(self):
        lib().mlkhip_release(self.handle)


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    if state.call(*state.args) != 0:
        raise RuntimeError(last_error())
    return state.out


def work(case):
    c, kind = case, case["kind"]
    if kind == "softmax":
        e = c["rows"] * c["cols"]
        return {"bytes": 2 * e * BYTES[c["dtype"]], "flops": 5 * e}
    if kind == "chain":
        return {"bytes": 2 * c["n"] * BYTES[c["dtype"]], "flops": 4 * c["n"]}
    if kind == "broadcast":
        e, b = c["rows"] * c["cols"], BYTES[c["dtype"]]
        return {"bytes": e * (b + 4) + c["cols"] * b, "flops": 4 * e}
    if kind == "gemm":
        m, k, n, out = c["m"], c["k"], c["n"], 8 if c["dtype"] == "f64" else 4
        return {"bytes": (m * k + k * n) * BYTES[c["dtype"]] + m * n * out * (2 if c["call"] else 1),
                "flops": 2 * m * k * n}
    b, s, d = c["batch"], c["seq"], c["dim"]
    return {"bytes": 2 * b * s * d * 2 + 4 * s + 4 * b * s * s, "flops": 2 * b * s * s * d + 7 * b * s * s}


def tolerance(case):
    """About four times the error measured against `exact` (its sums in 64
    bits), over the ranges of `draw`."""
    kind, dtype = case["kind"], case.get("dtype", "f32")
    if dtype == "f16" and kind in ("softmax", "chain"):
        return {"rel": 1e-3, "max": 4e-3}
    if dtype == "f64":
        return {"rel": 1e-14, "max": 1e-12}
    if kind == "gemm":
        # f32 sums of k products: 1.1e-6 measured at k = 4096, in k order.
        return {"rel": max(5e-7, 6.5e-8 * math.sqrt(case["k"]))}
    if kind == "score":
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 4e-7, "max": 4e-6}


def _softmax(x):
    e = torch.exp(x - x.amax(dim=1, keepdim=True))
    return e / e.sum(dim=1, keepdim=True)


def exact(case, seed):
    c, kind = case, case["kind"]
    ins, shape, _, first = _inputs(c, seed)
    x = ins[0].double()
    if kind == "softmax":
        return _softmax(x)
    if kind == "chain":
        return torch.sin(x * x + 3.0 * x) if c["op"] == "sin" else torch.exp(-0.5 * (x * x)) * x
    if kind == "broadcast":
        return torch.exp(0.5 * x + ins[1].double()) * x
    if kind == "gemm":
        ab = x @ ins[1].double()
        return ab if first is None else first.double() + ab
    out = torch.empty(shape, device="cuda", dtype=torch.float64)
    s = c["seq"]
    for b in range(c["batch"]):
        kt = ins[1][b].double().t().contiguous()
        scores = x[b] @ kt / math.sqrt(c["dim"]) + ins[2].double()
        out[b * s:(b + 1) * s] = _softmax(scores)
    return out
