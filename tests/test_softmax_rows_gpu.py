"""Softmax rows held in registers over several waves (softmaxRowWide: f32 rows
past 8192 columns, f16 rows; softmaxWaveRowScalar past 4096 columns), at the
edges of their ranges, against the oracle's f64 softmax.

Bounds: f32 results of f64 arithmetic round once, so each is within 1 ULP of
the oracle's value (2^-23 of it), or 2^-149 of a subnormal one; f16 results are
the oracle's rounded once (the polynomial's 1.9e-14 moves none here). The f32 arithmetic of the shorter rows
is held to the class's 1e-6."""
import numpy as np
import pytest

import oracle
from mlk2_amd import fixtures as fx
from mlk2_amd.backend import Binding, DeviceBuffer, lib

pytestmark = pytest.mark.gpu
LOWEST = {"f32": -3.4028234663852886e38, "f16": -65504.0}
NP = {"f32": np.float32, "f16": np.float16}


def rows_of(m, n, dtype):
    x = np.random.default_rng(m * 7919 + n).normal(0.0, 2.0, (m, n)).astype(NP[dtype])
    if m >= 9:
        x[1, :] = -np.inf                            # NaN row
        x[2, n // 2] = np.nan
        x[3, n - 1] = np.inf
        x[4, :] = LOWEST[dtype]                      # a row of the lowest value, -inf among it
        x[4, ::3] = -np.inf
        x[5, : n - n // 3] = LOWEST[dtype]           # masked but for its last third
        x[6, ::2] = -np.inf
        x[7] *= NP[dtype](5e9 if dtype == "f32" else 6e3)    # gaps far past exp's range
        x[8, 0] = NP[dtype](900.0)                   # all others underflow
    return x


def check(got, x, dtype, tight=True):
    ref = oracle.run(fx.softmax_call_module(*x.shape, "f64"), {0: x.astype(np.float64).reshape(-1)},
                     hw_threads=8)[1].reshape(x.shape)
    got = np.asarray(got, np.float64).reshape(x.shape)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    fin = ~np.isnan(ref)
    if dtype == "f16":
        with np.errstate(invalid="ignore"):
            want = ref.astype(np.float16).astype(np.float64)
        assert np.array_equal(got[fin], want[fin])
    elif tight:
        assert (np.abs(got[fin] - ref[fin]) <= 2.0 ** -23 * ref[fin] + 2.0 ** -149).all()
    else:
        assert (np.abs(got[fin] - ref[fin]) <= 1e-6).all()


@pytest.mark.parametrize("dtype,m,n", [("f32", 11, 8193), ("f32", 9, 16384), ("f32", 10, 16385), ("f32", 9, 32769),
                                       ("f32", 9, 65536), ("f32", 2, 65537), ("f32", 1, 40000),
                                       ("f16", 9, 15), ("f16", 11, 16), ("f16", 13, 23), ("f16", 9, 512),
                                       ("f16", 9, 1027), ("f16", 10, 2049), ("f16", 9, 4097), ("f16", 9, 16385),
                                       ("f16", 9, 65536), ("f16", 2, 65537)])
def test_register_rows(hip, dtype, m, n):
    x = rows_of(m, n, dtype)
    art = hip.build(fx.softmax_call_module(m, n, dtype))
    wide = 16 <= n <= 65536
    assert art.step_kernel_name(0).startswith("softmaxRowWide" if wide else "softmaxBlockRow")
    check(art.run({0: x.reshape(-1)})[1], x, dtype)


@pytest.mark.parametrize("n", [4097, 6001, 8190, 8191])
def test_scalar_rows_over_four_waves(hip, n):
    x = rows_of(11, n, "f32")
    art = hip.build(fx.softmax_call_module(11, n, "f32"))
    assert art.step_kernel_name(0) == "softmaxWaveRowScalar<32>"
    check(art.run({0: x.reshape(-1)})[1], x, "f32", tight=False)


def large_rows(n):
    """Finite maxima from where exp's arguments need more than 53 bits of x *
    log2(e) up to the largest float, of either sign, and constant rows."""
    x = np.zeros((13, n), np.float32)
    for r, v in enumerate([1e7, 1e19, 1e20, 1e25, 1e30, np.finfo(np.float32).max]):
        x[r, n // 3] = v
        x[6 + r] = -2.0 * v if v < 1e38 else -v
        x[6 + r, n - 1] = -v if v < 1e38 else -v / 2
    x[12] = np.float32(2.0 ** 84)
    return x


@pytest.mark.parametrize("n,skip", [(9000, 0), (9000, 3), (20000, 0), (65536, 0)])
@pytest.mark.parametrize("in_place", [False, True])
def test_rows_of_large_values(hip, n, skip, in_place):
    x = large_rows(n)
    art = hip.build(fx.softmax_call_module(*x.shape, "f32"))
    xb = _At(x, "f32", skip)
    yb = xb if in_place else _At(np.zeros_like(x), "f32", skip)
    art.run_device({0: xb, 1: yb})
    check(yb.values(), x, "f32")


# Of a row of two values every term but one has the same polynomial error: the
# results are the exact ones rounded once. 1.9e-14 of the term, as much of the sum
# and 2e-14 of its additions, against half an ULP of 2^-25 or more, are below
# 2^-18 of that half. With terms off by 2.5e-9 some 6% of them round elsewhere.
@pytest.mark.parametrize("n", [8200, 20000, 65535])
def test_rows_of_two_values(hip, n):
    c = np.random.default_rng(n).uniform(0.0, 12.0, 200).astype(np.float32)
    x = np.repeat(-c[:, None], n, axis=1)
    x[:, 0] = 0.0
    got = np.asarray(hip.build(fx.softmax_call_module(*x.shape, "f32")).run({0: x.reshape(-1)})[1]).reshape(x.shape)
    assert (got[:, 1:] == got[:, 1:2]).all()
    e = np.exp(-c.astype(np.float64))
    for have, ref in ((got[:, 0], 1 / (1 + (n - 1) * e)), (got[:, 1], e / (1 + (n - 1) * e))):
        half = np.spacing(ref.astype(np.float32)).astype(np.float64) / 2
        assert (np.abs(have - ref) <= half * (1 + 2.0 ** -18)).all()


class _At:
    """A device buffer bound `skip` elements into its allocation."""

    def __init__(self, x, dtype, skip):
        pad = np.zeros(skip + x.size + 16, NP[dtype])
        pad[skip:skip + x.size] = x.reshape(-1)
        self.buf, self.skip, self.n = DeviceBuffer.from_array(pad, dtype), skip, x.size

    def binding(self):
        return Binding(self.buf.ptr + self.skip * (self.buf.nbytes // self.buf.elements), self.n, self.buf.code, 0)

    def values(self):
        return self.buf.to_numpy()[self.skip:self.skip + self.n]


@pytest.mark.parametrize("dtype,n,skips", [("f32", 9001, (1, 1)), ("f32", 9001, (3, 2)), ("f32", 9000, (2, 2)),
                                           ("f16", 77, (5, 5)), ("f16", 77, (1, 0)), ("f16", 3000, (7, 7))])
def test_rows_off_16_bytes(hip, dtype, n, skips):
    # x and y off 16 bytes by the same amount run in registers; by different
    # ones on the general kernel. Nothing beside y is written.
    x = rows_of(9, n, dtype)
    xb, yb = _At(x, dtype, skips[0]), _At(np.zeros_like(x), dtype, skips[1])
    hip.build(fx.softmax_call_module(9, n, dtype)).run_device({0: xb, 1: yb})
    check(yb.values(), x, dtype)
    whole = yb.buf.to_numpy()
    assert not whole[:skips[1]].any() and not whole[skips[1] + x.size:].any()


@pytest.mark.parametrize("dtype,n", [("f32", 20000), ("f16", 300), ("f16", 5000)])
def test_rows_in_place(hip, dtype, n):
    x = rows_of(9, n, dtype)
    b = DeviceBuffer.from_array(x.reshape(-1), dtype)
    hip.build(fx.softmax_call_module(9, n, dtype)).run_device({0: b, 1: b})
    check(b.to_numpy(), x, dtype)


def test_rows_past_one_grid(hip):
    # 2^26 rows of 16: their workgroups are more threads than one launch holds.
    m, n = (1 << 26) + 5, 16
    art = hip.build(fx.softmax_call_module(m, n, "f16"))
    assert art.step_kernel_name(0).startswith("softmaxRowWide")
    xb, yb = DeviceBuffer(m * n, "f16"), DeviceBuffer(m * n, "f16")
    plain = np.tile(np.array([1.0, 2.0], np.float16), n // 2)
    assert lib().mlkhip_fill32(xb.ptr, int(plain[:2].view(np.uint32)[0]), xb.nbytes) == 0
    yb.fill_zero()
    at = [0, 1, (1 << 25) - 1, 1 << 25, (1 << 26) - 1, 1 << 26, m - 1]   # ends of launches and of the rows
    x = rows_of(len(at), n, "f16")
    for r, row in zip(at, x):
        assert lib().mlkhip_memcpy_h2d(xb.ptr + r * n * 2, row.ctypes.data, n * 2) == 0
    art.run_device({0: xb, 1: yb})
    got = yb.to_numpy().reshape(m, n)
    check(got[at], x, "f16")
    rest = got[2].copy()
    check(rest, plain.reshape(1, n), "f16")
    same = (got.view(np.uint64) == rest.view(np.uint64)).all(axis=1)
    assert same.sum() == m - len(at) and not same[at].any()
