"""GEMM shapes off the whole blocks of the MFMA forms (the ragged members of
gemmF16Dma8s, tiles of 128 and 256, and of gemmF32Dma): edges of tiles, of K
steps and of the 16-byte pieces, against the f64 product.

Bound: a sum of k products in precision u = 2^-24, in any order, is within
(k + 2) u sum |a||b| of the exact one; the f64 product the results are held to
adds (k + 2) 2^-53 of it."""
import numpy as np
import pytest

import oracle
from mlk2_amd import fixtures as fx
from mlk2_amd.backend import Binding, DeviceBuffer
from test_score_two_pass_gpu import _Capture

pytestmark = pytest.mark.gpu
NP = {"f16": np.float16, "f32": np.float32}
KERNEL = {"f16": "gemmF16Dma8s", "f32": "gemmF32Dma"}
U = 2.0 ** -24


def operands(m, k, n, dtype):
    rng = np.random.default_rng(m * 31 + k * 17 + n)
    return (rng.uniform(-1, 1, (m, k)).astype(NP[dtype]), rng.uniform(-1, 1, (k, n)).astype(NP[dtype]),
            rng.uniform(-1, 1, (m, n)).astype(np.float32))


def module(m, k, n, dtype, call):
    km = fx.matmul_call_module(m, k, n, dtype)
    return km if call else fx.synth_gemm(km)


def check(got, a, b, c, call):
    a, b, c = a.astype(np.float64), b.astype(np.float64), c.astype(np.float64)
    ref, size = a @ b, np.abs(a) @ np.abs(b)
    if call:
        ref, size = ref + c, size + np.abs(c)
    got = np.asarray(got, np.float64).reshape(ref.shape)
    bound = (a.shape[1] + 3) * (U + 2.0 ** -53) * size
    assert (np.abs(got - ref) <= bound).all(), float((np.abs(got - ref) / np.maximum(bound, 1e-300)).max())


# f16: K steps of 32 (one partial, one whole, 3 mod 4), rows and columns one
# past and one short of a tile, aligned rows and copied ones (k or n off 8),
# enough tiles for tiles of 256. f32: K steps of 64.
@pytest.mark.parametrize("call", [False, True])
@pytest.mark.parametrize("dtype,m,k,n", [
    ("f16", 1020, 16, 1016), ("f16", 127, 32, 264), ("f16", 200, 24, 250), ("f16", 130, 40, 128), ("f16", 128, 100, 257),
    ("f16", 1025, 104, 1000), ("f16", 1000, 999, 1001), ("f16", 1000, 1000, 1003), ("f16", 1001, 227, 1000),
    ("f16", 3900, 520, 4040), ("f16", 3841, 545, 3847),
    ("f32", 190, 12, 190), ("f32", 63, 64, 127), ("f32", 130, 100, 66), ("f32", 129, 65, 131), ("f32", 1000, 196, 900),
    ("f32", 700, 1001, 999)])
def test_edges(hip, dtype, m, k, n, call):
    a, b, c = operands(m, k, n, dtype)
    art = hip.build(module(m, k, n, dtype, call))
    assert art.step_kernel_name(0) == f"{KERNEL[dtype]}<{'true' if call else 'false'}>"
    got = art.run({0: a.reshape(-1), 1: b.reshape(-1), 2: c.reshape(-1)})[2]
    check(got, a, b, c, call)


@pytest.mark.parametrize("dtype,m,k,n", [("f16", 300, 104, 264), ("f16", 300, 99, 257), ("f16", 3900, 520, 4040),
                                         ("f32", 200, 101, 130), ("f32", 200, 100, 132)])
def test_non_finite_columns_skip_zeros(hip, dtype, m, k, n):
    # Call(MatMul) leaves out A[i,p] == 0, also against an inf or NaN of B: the
    # waves that meet one recompute their part of C in order, within bounds.
    a, b, c = operands(m, k, n, dtype)
    a[:, 5] = 0
    a[7, 5] = a[m - 1, 5] = 0.5
    b[5, 2], b[5, n - 1] = np.inf, np.nan
    art = hip.build(module(m, k, n, dtype, True))
    assert art.step_kernel_name(0) == f"{KERNEL[dtype]}<true>"
    got = art.run({0: a.reshape(-1), 1: b.reshape(-1), 2: c.reshape(-1)})[2].reshape(m, n)
    rows = sorted({0, 7, m // 2, m - 1})
    ref = oracle.run(fx.matmul_call_module(len(rows), k, n, "f64", "f64"),
                     {0: a[rows].astype(np.float64).reshape(-1), 1: b.astype(np.float64).reshape(-1)},
                     init={2: c[rows].astype(np.float64).reshape(-1)})[2].reshape(len(rows), n)
    part = got[rows]
    assert np.array_equal(np.isnan(part), np.isnan(ref)) and np.array_equal(np.isinf(part), np.isinf(ref))
    assert np.isfinite(np.delete(got, [7, m - 1], 0)).all()
    fin = np.isfinite(ref)
    size = np.abs(a[rows].astype(np.float64)) @ np.where(np.isfinite(b), np.abs(b), 0).astype(np.float64)
    assert (np.abs(part[fin] - ref[fin]) <= ((k + 3) * (U + 2.0 ** -53) * (size + np.abs(c[rows])))[fin]).all()


# One infinity in B: 15 times the finite product's time (206, with one row and
# one step's loads at a time).
def test_non_finite_products_stay_fast(hip):
    n = 1000
    a, b, c = operands(n, n, n, "f32")
    art = hip.build(module(n, n, n, "f32", True))
    bufs = {0: DeviceBuffer.from_array(a, "f32"), 1: DeviceBuffer.from_array(b, "f32"), 2: DeviceBuffer.from_array(c, "f32")}
    finite = art.time_device_span(bufs, 10)
    b[n // 2, n // 3] = np.inf
    bufs[1] = DeviceBuffer.from_array(b, "f32")
    assert art.time_device_span(bufs, 3, 1) <= 60 * finite


class _At:
    def __init__(self, x, dtype, skip):
        pad = np.zeros(skip + x.size + 8, NP[dtype])
        pad[skip:skip + x.size] = x.reshape(-1)
        self.buf, self.skip, self.n = DeviceBuffer.from_array(pad, dtype), skip, x.size

    def binding(self):
        return Binding(self.buf.ptr + self.skip * (self.buf.nbytes // self.buf.elements), self.n, self.buf.code, 0)


@pytest.mark.parametrize("dtype,m,k,n", [("f16", 300, 104, 264), ("f32", 200, 100, 132), ("f16", 1000, 600, 1000)])
def test_operands_at_any_element(hip, dtype, m, k, n):
    # Bases off 16 bytes are copied to aligned rows; nothing beside C is written.
    a, b, c = operands(m, k, n, dtype)
    cb = _At(c, "f32", 3)
    hip.build(module(m, k, n, dtype, True)).run_device({0: _At(a, dtype, 1), 1: _At(b, dtype, 3), 2: cb})
    whole = cb.buf.to_numpy()
    check(whole[3:3 + c.size], a, b, c, True)
    assert not whole[:3].any() and not whole[3 + c.size:].any()


def test_allocation_free_entry_without_room(hip):
    # Copies past the array's 32 MiB: the general kernel runs, within the bound.
    m, k, n = 3001, 3001, 3001
    a, b, c = operands(m, k, n, "f16")
    art = hip.build(module(m, k, n, "f16", False))
    ab, bb = DeviceBuffer.from_array(a, "f16"), DeviceBuffer.from_array(b, "f16")
    y = DeviceBuffer(m * n, "f32")
    art.run_device_noalloc({0: ab, 1: bb, 2: y})
    check(y.to_numpy(), a, b, c, False)


def test_captured_workspace_outlives_a_larger_one(hip):
    # A graph holds the workspace of A's copy; a run that copies B too asks for
    # a larger one, and the graph's stays until the artifact is released.
    m, k, n = 300, 104, 264
    a, b, c = operands(m, k, n, "f16")
    art = hip.build(module(m, k, n, "f16", False))
    off, even, odd = _At(a, "f16", 1), _At(b, "f16", 0), _At(b, "f16", 3)
    out, eager = DeviceBuffer(m * n, "f32"), DeviceBuffer(m * n, "f32")
    cap = _Capture()
    stream = cap.stream.value

    def run(bound, y):
        art.run_device({0: off, 1: bound, 2: y}, stream=stream, sync=False)
        cap("hipStreamSynchronize", cap.stream)
        check(y.to_numpy(), a, b, c, False)

    run(even, eager)
    with cap:
        art.run_device({0: off, 1: even, 2: out}, stream=stream, sync=False)
    run(odd, eager)
    others = [DeviceBuffer.from_array(np.full(m * 128, 3.0), "f16") for _ in range(8)]
    for bound in (odd, even, odd):
        cap.replay()
        check(out.to_numpy(), a, b, c, False)
        run(bound, eager)
    for other in others:
        assert (other.to_numpy() == 3.0).all()
    cap.close()
