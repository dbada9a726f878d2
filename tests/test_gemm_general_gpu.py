"""The general GEMM on matrix cores (gemmGeneral: operands straight from
global memory) at the edges of its tiles, vectors, K steps and K ranges, against
the f64 product.

Bound: a sum of k products in precision u, in any order, is within
(k + 2) u sum |a||b| of the exact one (u = 2^-24 for f16 and f32 operands,
whose f16 products are exact in f32; 2^-53 for f64); the f64 product the results
are held to adds its own (k + 2) 2^-53 share."""
import ctypes

import numpy as np
import pytest

import oracle
from mlk2_amd import fixtures as fx
from mlk2_amd.backend import DTYPE_CODE, Binding, DeviceBuffer, lib

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


class _Gemm(ctypes.Structure):
    """mlkd_gemm of csrc/device_abi.h."""
    _fields_ = [("a", ctypes.c_void_p), ("b", ctypes.c_void_p), ("c", ctypes.c_void_p),
                ("a_dtype", ctypes.c_int32), ("b_dtype", ctypes.c_int32), ("c_dtype", ctypes.c_int32),
                ("accumulate", ctypes.c_int32), ("m", ctypes.c_int64), ("n", ctypes.c_int64), ("k", ctypes.c_int64),
                ("lda", ctypes.c_int64), ("ldb", ctypes.c_int64), ("ldc", ctypes.c_int64), ("variant", ctypes.c_int32),
                ("skip_zero_a", ctypes.c_int32), ("pad_", ctypes.c_int32), ("work", ctypes.c_void_p),
                ("work_bytes", ctypes.c_int64)]


def tile(m, k, n, dtype, call):
    """The output tile of a workgroup. 16, 32 or 64 rows (64 also the scalar
    kernel's) by 16 16-byte pieces of columns: the direct kernel's."""
    d, rows, cols = DTYPE_CODE[dtype], ctypes.c_int64(), ctypes.c_int64()
    p = _Gemm(None, None, None, d, d, DTYPE_CODE["f64" if dtype == "f64" else "f32"], call, m, n, k, k, n, n, -1, call)
    lib().mlkd_gemm_tile(ctypes.byref(p), ctypes.byref(rows), ctypes.byref(cols))
    return rows.value, cols.value


# Two and four row tiles to a workgroup (enough tiles for the chip), one, two
# and four waves, rows and columns off the tiles, K off its steps.
SEVERAL = [("f64", 769, 200, 767, 2), ("f64", 2047, 100, 1025, 4), ("f64", 4095, 40, 1023, 4), ("f32", 17003, 50, 13, 2),
           ("f32", 32771, 50, 13, 4), ("f16", 17003, 70, 60, 2), ("f16", 32771, 70, 60, 4)]


@pytest.mark.parametrize("call", [False, True])
@pytest.mark.parametrize("dtype,m,k,n,tiles", SEVERAL)
def test_several_row_tiles(hip, dtype, m, k, n, tiles, call):
    a, b, c = operands(m, k, n, dtype)
    assert tile(m, k, n, dtype, call) == (16 * tiles, 16 * V[dtype])
    art = hip.build(module(m, k, n, dtype, call))
    check(art.run({0: a.reshape(-1), 1: b.reshape(-1), 2: c.reshape(-1)})[2], a, b, c, dtype, call)


def check_skip(got, a, b, c, dtype):
    """Call(MatMul), which leaves out A[i,p] == 0, also against an inf or NaN of B."""
    a, b, c = a.astype(np.float64), b.astype(np.float64), c.astype(np.float64)
    finite = np.where(np.isfinite(b), b, 0)
    ref, size = a @ finite + c, np.abs(a) @ np.abs(finite) + np.abs(c)
    for p, j in np.argwhere(~np.isfinite(b)):
        on = a[:, p] != 0
        ref[on, j] += a[on, p] * b[p, j]
    got = np.asarray(got, np.float64).reshape(ref.shape)
    for kind in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(kind(got), kind(ref))
    fin = np.isfinite(ref)
    assert (np.abs(got[fin] - ref[fin]) <= ((a.shape[1] + 3) * (U[dtype] + 2.0 ** -53) * size)[fin]).all()


# And over K ranges, with K off the steps that are read together (16, 8).
@pytest.mark.parametrize("dtype,m,k,n", [c[:4] for c in SEVERAL] + [("f64", 5, 4099, 70), ("f64", 300, 71, 500),
                                                                   ("f32", 300, 203, 300), ("f16", 200, 701, 300)])
def test_non_finite_columns_over_tiles(hip, dtype, m, k, n):
    a, b, c = operands(m, k, n, dtype)
    a[:, 5] = a[:, k - 1] = 0
    a[[0, m // 2, m - 1], 5] = 0.5
    a[m - 1, k - 1] = -1
    b[5, 2], b[5, n - 1], b[k - 1, n // 2] = np.inf, np.nan, np.inf
    art = hip.build(module(m, k, n, dtype, True))
    check_skip(art.run({0: a.reshape(-1), 1: b.reshape(-1), 2: c.reshape(-1)})[2], a, b, c, dtype)


# A non-finite product adds each element of some tiles up in order: 7 times the
# finite one's time here (38, with a step's loads waited for at each step).
def test_non_finite_products_stay_fast(hip):
    n = 1024
    rng = np.random.default_rng(3)
    art = hip.build(module(n, n, n, "f64", True))
    b = rng.uniform(-1, 1, (n, n))
    bufs = {0: DeviceBuffer.from_array(rng.uniform(-1, 1, (n, n)), "f64"), 1: DeviceBuffer.from_array(b, "f64"),
            2: DeviceBuffer.from_array(np.zeros(n * n), "f64")}
    finite = art.time_device_span(bufs, 10)
    b[n // 2, n // 3] = np.inf
    bufs[1] = DeviceBuffer.from_array(b, "f64")
    assert art.time_device_span(bufs, 3, 1) <= 20 * finite


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
