"""The general GEMM on matrix cores (gemmGeneral: operands straight from
global memory) at the edges of its tiles, vectors, K steps and K ranges, against
the f64 product.

Bound: a sum of k products in precision u, in any order, is within
(k + 2) u sum |a||b| of the exact one (u = 2^-24 for f16 and f32 operands,
whose f16 products are exact in f32; 2^-53 for f64); the f64 product the results
are held to adds its own (k + 2) 2^-53 share."""
import numpy as np
import pytest

import oracle
from mlk2_amd import fixtures as fx
from mlk2_amd.backend import Binding, DeviceBuffer

pytestmark = pytest.mark.gpu
NP = {"f16": np.float16, "f32": np.float32, "f64": np.float64}
U = {"f16": 2.0 ** -24, "f32": 2.0 ** -24, "f64": 2.0 ** -53}
V = {"f16": 8, "f32": 4, "f64": 2}


def operands(m, k, n, dtype, seed=0):
    rng = np.random.default_rng(seed + m * 31 + k * 17 + n)
    a = rng.uniform(-1, 1, (m, k)).astype(NP[dtype])
    b = rng.uniform(-1, 1, (k, n)).astype(NP[dtype])
    if dtype == "f16" and k > 2:    # subnormals count
        a[:, 1] = np.float16(6e-8)
    c = rng.uniform(-1, 1, (m, n))
    return a, b, (c if dtype == "f64" else c.astype(np.float32))


def module(m, k, n, dtype, call):
    km = fx.matmul_call_module(m, k, n, dtype, "f64" if dtype == "f64" else "f32")
    return km if call else fx.synth_gemm(km)


def check(got, a, b, c, dtype, call):
    a, b, c = a.astype(np.float64), b.astype(np.float64), c.astype(np.float64)
    ref, size = a @ b, np.abs(a) @ np.abs(b)
    if call:
        ref, size = ref + c, size + np.abs(c)
    got = np.asarray(got, np.float64).reshape(ref.shape)
    bound = (a.shape[1] + 3) * (U[dtype] + 2.0 ** -53) * size + 2.0 ** -149
    assert (np.abs(got - ref) <= bound).all(), float((np.abs(got - ref) / bound).max())


# Rows around 16, 32, 64; columns from one vector up, around a tile; K from
# one step up, around a step, and long enough for K ranges.
SIZES = [(1, 32, 8), (16, 32, 128), (17, 33, 129), (15, 63, 9), (33, 64, 127), (64, 100, 260), (65, 95, 60),
         (3, 4096, 1000), (16, 2100, 385), (31, 8191, 136), (200, 64, 17), (100, 3000, 8)]


@pytest.mark.parametrize("call", [False, True])
@pytest.mark.parametrize("m,k,n", SIZES)
@pytest.mark.parametrize("dtype", ["f16", "f32", "f64"])
def test_edges(hip, dtype, m, k, n, call):
    a, b, c = operands(m, k, n, dtype)
    art = hip.build(module(m, k, n, dtype, call))
    got = art.run({0: a.reshape(-1), 1: b.reshape(-1), 2: c.reshape(-1)})[2]
    check(got, a, b, c, dtype, call)


# Each XCD's share of the tiles, where 8 do not divide them: every tile once.
@pytest.mark.parametrize("tiles", [1, 7, 8, 9, 15, 17, 22, 27])
@pytest.mark.parametrize("m", [16, 40])
def test_numbers_of_tiles(hip, m, tiles):
    a, b, c = operands(m, 40, 32 * tiles - 1, "f64")
    got = hip.build(module(m, 40, 32 * tiles - 1, "f64", True)).run(
        {0: a.reshape(-1), 1: b.reshape(-1), 2: c.reshape(-1)})[2]
    check(got, a, b, c, "f64", True)


def test_names(hip):
    # Long K over few tiles: K ranges in several workgroups, then their sum.
    name = hip.build(module(16, 4096, 4096, "f16", False)).step_kernel_name(0)
    assert name == "gemmGeneral<float>+gemmSumParts<_Float16>"
    assert hip.build(module(512, 512, 512, "f64", False)).step_kernel_name(0) == "gemmGeneral<double>"
    # Below one K step or one vector of columns: the scalar kernel.
    for m, k, n in [(9, 31, 40), (9, 40, 7)]:
        a, b, c = operands(m, k, n, "f16")
        art = hip.build(module(m, k, n, "f16", False))
        assert art.step_kernel_name(0) in ("gemmGeneral<float>", "gemmF16Dma8s<false>")
        check(art.run({0: a.reshape(-1), 1: b.reshape(-1)})[2], a, b, c, "f16", False)


@pytest.mark.parametrize("dtype", ["f16", "f32", "f64"])
@pytest.mark.parametrize("k", [200, 5000])
def test_non_finite_columns_skip_zeros(hip, dtype, k):
    # Call(MatMul) leaves out A[i,p] == 0, also against an inf or NaN of B.
    m, n = 18, 3 * V[dtype] + 1
    a, b, c = operands(m, k, n, dtype)
    a[:, 5] = 0
    a[7, 5] = 0.5
    b[5, 2], b[5, n - 1] = np.inf, np.nan
    art = hip.build(module(m, k, n, dtype, True))
    got = art.run({0: a.reshape(-1), 1: b.reshape(-1), 2: c.reshape(-1)})[2].reshape(m, n)
    ref = oracle.run(fx.matmul_call_module(m, k, n, "f64", "f64"), {0: a.astype(np.float64).reshape(-1),
                     1: b.astype(np.float64).reshape(-1)}, init={2: c.astype(np.float64).reshape(-1)})[2].reshape(m, n)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    fin = np.isfinite(ref)
    size = np.abs(a.astype(np.float64)) @ np.where(np.isfinite(b), np.abs(b), 0).astype(np.float64) + np.abs(c)
    assert (np.abs(got[fin] - ref[fin]) <= ((k + 3) * (U[dtype] + 2.0 ** -53) * size)[fin]).all()


class _At:
    def __init__(self, x, dtype, skip):
        pad = np.zeros(skip + x.size + 8, NP[dtype])
        pad[skip:skip + x.size] = x.reshape(-1)
        self.buf, self.skip, self.n = DeviceBuffer.from_array(pad, dtype), skip, x.size

    def binding(self):
        return Binding(self.buf.ptr + self.skip * (self.buf.nbytes // self.buf.elements), self.n, self.buf.code, 0)


@pytest.mark.parametrize("dtype", ["f16", "f32", "f64"])
@pytest.mark.parametrize("m,k,n", [(8, 512, 512), (5, 1029, 77)])
def test_operands_at_any_element(hip, dtype, m, k, n):
    # Bases off 16 bytes; nothing beside C is written.
    out = "f64" if dtype == "f64" else "f32"
    a, b, c = operands(m, k, n, dtype)
    cb = _At(c, out, 3)
    hip.build(module(m, k, n, dtype, True)).run_device({0: _At(a, dtype, 1), 1: _At(b, dtype, 3), 2: cb})
    whole = cb.buf.to_numpy()
    check(whole[3:3 + c.size], a, b, c, dtype, True)
    assert not whole[:3].any() and not whole[3 + c.size:].any()


@pytest.mark.parametrize("dtype", ["f16", "f64"])
def test_allocation_free_entry_agrees(hip, dtype):
    m, k, n = 16, 4096, 640
    a, b, c = operands(m, k, n, dtype)
    art = hip.build(module(m, k, n, dtype, False))
    out = "f64" if dtype == "f64" else "f32"
    ab, bb = DeviceBuffer.from_array(a, dtype), DeviceBuffer.from_array(b, dtype)
    y, z = DeviceBuffer(m * n, out), DeviceBuffer(m * n, out)
    art.run_device({0: ab, 1: bb, 2: y})
    art.run_device_noalloc({0: ab, 1: bb, 2: z})
    assert np.array_equal(y.to_numpy().view(np.uint8), z.to_numpy().view(np.uint8))
    check(y.to_numpy(), a, b, c, dtype, False)
