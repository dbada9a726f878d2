"""Score-softmax in two passes: head dims 64 and 128, sequences of one 128-key
panel (from four at dim 64) up to several per key range, uneven ranges, padded
sequences, S off 16 bytes, masked keys, and rows whose largest score is far
from 0, against the f64 softmax.

Bound: with u = 2^-24, a score in f32 (a sum of dim products, the scale, the
bias, three roundings) is within e = u ((dim + 4) sum |q k| / div + 4 |bias| + 2
|score - shift|) of the exact one; a weight, exp(score) over a sum of seq of
them with one-ulp exponentials, within 2 max(e) + (seq + 8) u, relatively."""
import ctypes

import numpy as np
import pytest

from mlk2_amd import fixtures as fx
from mlk2_amd.backend import Binding, DeviceBuffer

pytestmark = pytest.mark.gpu
U = 2.0 ** -24
TWO_PASS = "scoreStatsQ+scoreStoreQ"


def operands(b, s, d, scale=1.0):
    rng = np.random.default_rng(b * 7919 + s * 31 + d)
    q, k = (rng.standard_normal((b, s, d)).astype(np.float16) for _ in range(2))
    return (q * np.float16(scale)).astype(np.float16), k, (0.1 * rng.standard_normal(s)).astype(np.float32)


def check(got, q, k, bias):
    b, s, d = q.shape
    q, k, bias = q.astype(np.float64), k.astype(np.float64), bias.astype(np.float64)
    kt = np.swapaxes(k, 1, 2)
    x = q @ kt / np.sqrt(d) + bias
    live = np.isfinite(bias) & (bias > -1e30)
    top = x.max(axis=2, keepdims=True)
    with np.errstate(invalid="ignore"):
        e = np.exp(x - top)
    ref = e / e.sum(axis=2, keepdims=True)
    size = np.abs(q) @ np.abs(kt) / np.sqrt(d)
    err = U * ((d + 4) * size + 4 * np.abs(np.where(live, bias, 0)) + 2 * np.abs(np.where(live, x - top, 0)) +
               2 * np.abs(top))
    rel = 2 * np.where(live, err, 0).max(axis=2, keepdims=True) + (s + 8) * U
    got = np.asarray(got, np.float64).reshape(ref.shape)
    assert (np.abs(got - ref) <= rel * ref + 2.0 ** -125).all(), float((np.abs(got - ref) / (rel * ref + 2.0 ** -125)).max())


def built(hip, b, s, d):
    art = hip.build(fx.score_softmax_module(b, s, d))
    assert art.step_kernel_name(0) == TWO_PASS
    return art


# Ranges from one to eight, the last one shorter (384, 896, 1152, 2176), one for
# many batches (40); padded lengths (dim 128 only), a multiple of 4 and not.
@pytest.mark.parametrize("b,s,d", [
    (5, 128, 128), (2, 512, 64), (2, 384, 128), (3, 896, 64), (40, 896, 64), (1, 1024, 64), (9, 1024, 128),
    (3, 1152, 128), (1, 2048, 64), (1, 2176, 128), (2, 129, 128), (3, 500, 128), (1, 1030, 128)])
def test_shapes(hip, b, s, d):
    q, k, bias = operands(b, s, d)
    check(built(hip, b, s, d).run({0: q.reshape(-1), 1: k.reshape(-1), 2: bias})[3], q, k, bias)


# Masked panels, ranges and single keys (-inf and the lowest float), and scores
# far above and below 0 and spread widely.
@pytest.mark.parametrize("b,s,d", [(2, 512, 64), (1, 1024, 128), (1, 2048, 64), (2, 300, 128)])
@pytest.mark.parametrize("kind", ["inf", "lowest", "all", "tail", "high", "low", "wide"])
def test_masks_and_magnitudes(hip, b, s, d, kind):
    q, k, bias = operands(b, s, d, 16.0 if kind == "wide" else 1.0)
    if kind in ("inf", "lowest"):
        bias[np.arange(s) % 3 == 1] = -np.inf if kind == "inf" else np.finfo(np.float32).min
        bias[: s // 2] = -np.inf if kind == "inf" else np.finfo(np.float32).min
    elif kind == "all":
        bias[:] = np.finfo(np.float32).min
    elif kind == "tail":
        bias[5:] = -np.inf
    elif kind != "wide":
        bias += np.float32(300.0 if kind == "high" else -300.0)
    check(built(hip, b, s, d).run({0: q.reshape(-1), 1: k.reshape(-1), 2: bias})[3], q, k, bias)


@pytest.mark.parametrize("b,s,d", [(2, 512, 64), (1, 500, 128)])
def test_no_live_key_and_nan(hip, b, s, d):
    q, k, bias = operands(b, s, d)
    art = built(hip, b, s, d)
    assert np.isnan(np.asarray(art.run({0: q.reshape(-1), 1: k.reshape(-1), 2: np.full(s, -np.inf, np.float32)})[3])).all()
    q[0, 7, 3] = np.nan
    got = np.asarray(art.run({0: q.reshape(-1), 1: k.reshape(-1), 2: bias})[3]).reshape(b, s, s)
    assert np.isnan(got[0, 7]).all() and np.isnan(got).sum() == s


# A row's weights add up to 1 but for the rounding of 1 / sum, at most u, evenly
# spread (u / sqrt(3) rms), and of the weights, at most 2 u of each, by chance (2 u
# sqrt(sum of p^2)); sums in f32 are off by twice that.
@pytest.mark.parametrize("b,s", [(16, 512), (3, 640), (8, 1024), (2, 2048), (1, 8192)])
def test_row_sums_at_dim_64(hip, b, s):
    q, k, bias = operands(b, s, 64)
    p = np.asarray(built(hip, b, s, 64).run({0: q.reshape(-1), 1: k.reshape(-1), 2: bias})[3], np.float64).reshape(-1, s)
    off = p.sum(axis=1) - 1
    assert np.sqrt((off ** 2).mean()) <= U * (1 / np.sqrt(3) + 2 * np.sqrt((p ** 2).sum(axis=1).mean()))


# Masks past float's range in base 2 keep their order; +inf makes its row NaN.
def test_bias_at_the_ends_of_the_range_at_dim_64(hip):
    b, s = 2, 512
    q, k, bias = operands(b, s, 64)
    art = built(hip, b, s, 64)
    bias[:] = np.finfo(np.float32).min
    bias[[3, 130, 511]] = -2.5e38
    got = np.asarray(art.run({0: q.reshape(-1), 1: k.reshape(-1), 2: bias})[3]).reshape(-1, s)
    assert (got[:, [3, 130, 511]] == np.float32(1 / 3)).all()
    assert not np.delete(got, [3, 130, 511], 1).any()
    bias[7] = np.inf
    assert np.isnan(np.asarray(art.run({0: q.reshape(-1), 1: k.reshape(-1), 2: bias})[3])).all()


class _At:
    def __init__(self, n, skip):
        self.buf, self.skip, self.n = DeviceBuffer.from_array(np.zeros(n + 8, np.float32), "f32"), skip, n

    def binding(self):
        return Binding(self.buf.ptr + 4 * self.skip, self.n, self.buf.code, 0)


def device(q, k, bias):
    return {0: DeviceBuffer.from_array(q, "f16"), 1: DeviceBuffer.from_array(k, "f16"),
            2: DeviceBuffer.from_array(bias, "f32")}


@pytest.mark.parametrize("b,s,d", [(2, 512, 64), (1, 384, 128), (2, 300, 128)])
def test_output_at_any_element(hip, b, s, d):
    q, k, bias = operands(b, s, d)
    out = _At(b * s * s, 3)
    built(hip, b, s, d).run_device({**device(q, k, bias), 3: out})
    whole = out.buf.to_numpy()
    check(whole[3:3 + out.n], q, k, bias)
    assert not whole[:3].any() and not whole[3 + out.n:].any()


@pytest.mark.parametrize("b,s,d", [(2, 512, 64), (1, 1024, 128), (2, 300, 128)])
def test_allocation_free_entry(hip, b, s, d):
    q, k, bias = operands(b, s, d)
    art, bufs, out = built(hip, b, s, d), device(q, k, bias), [DeviceBuffer(b * s * s, "f32") for _ in range(2)]
    art.run_device({**bufs, 3: out[0]})
    art.run_device_noalloc({**bufs, 3: out[1]})
    assert np.array_equal(out[0].to_numpy(), out[1].to_numpy())


# Statistics past the entry's 32 MiB (two floats per row and key range): a step
# that has them in the workspace only runs without them.
def test_allocation_free_entry_without_room(hip):
    b, s, d = 8200, 256, 64
    art = hip.build(fx.score_softmax_module(b, s, d))
    q, k, bias = operands(1, s, d)
    bufs = device(np.broadcast_to(q, (b, s, d)), np.broadcast_to(k, (b, s, d)), bias)
    out = DeviceBuffer(b * s * s, "f32")
    art.run_device_noalloc({**bufs, 3: out})
    got = out.to_numpy().reshape(b, -1)
    check(got[-1], q, k, bias)
    assert (got == got[-1]).all()


class _Capture:
    """Captures what is enqueued on a new stream into a HIP graph (mode 0:
    nothing may allocate meanwhile, 2: relaxed)."""

    def __init__(self, mode=0):
        self.mode = mode
        with open("/proc/self/maps") as f:
            path = next(line.split()[-1] for line in f if "libamdhip64" in line)
        self.hip, self.stream, self.graph, self.exec = ctypes.CDLL(path), *(ctypes.c_void_p() for _ in range(3))
        self("hipStreamCreate", ctypes.byref(self.stream))

    def __call__(self, name, *args):
        assert getattr(self.hip, name)(*args) == 0, name

    def __enter__(self):
        self("hipStreamBeginCapture", self.stream, self.mode)
        return self.stream.value

    def __exit__(self, *exc):
        self("hipStreamEndCapture", self.stream, ctypes.byref(self.graph))
        self("hipGraphInstantiate", ctypes.byref(self.exec), self.graph, None, None, ctypes.c_size_t(0))

    def replay(self):
        self("hipGraphLaunch", self.exec, self.stream)
        self("hipStreamSynchronize", self.stream)

    def close(self):
        self("hipGraphExecDestroy", self.exec)
        self("hipGraphDestroy", self.graph)
        self("hipStreamDestroy", self.stream)


# A stream's first run, under capture: no workspace is allocated, and the step
# runs on the kernels that need none.
@pytest.mark.parametrize("case", ["score 2x512x64", "gemm f64 128"])
def test_first_run_under_capture(hip, case):
    if case.startswith("score"):
        q, k, bias = operands(2, 512, 64)
        art, bufs, n, dtype = hip.build(fx.score_softmax_module(2, 512, 64)), device(q, k, bias), 2 * 512 * 512, "f32"
    else:
        rng = np.random.default_rng(5)
        a, b = rng.uniform(-1, 1, (128, 4096)), rng.uniform(-1, 1, (4096, 128))
        art, n, dtype = hip.build(fx.synth_gemm(fx.matmul_call_module(128, 4096, 128, "f64", "f64"))), 128 * 128, "f64"
        bufs = {0: DeviceBuffer.from_array(a, "f64"), 1: DeviceBuffer.from_array(b, "f64")}
    out, eager = DeviceBuffer(n, dtype), DeviceBuffer(n, dtype)
    o = max(bufs) + 1
    cap = _Capture()
    with cap as stream:
        art.run_device({**bufs, o: out}, stream=stream, sync=False)
    for _ in range(3):
        cap.replay()
        art.run_device({**bufs, o: eager})
        for got in (out.to_numpy(), eager.to_numpy()):
            if case.startswith("score"):
                check(got, q, k, bias)
            else:
                assert (np.abs(got.reshape(128, 128) - a @ b) <= 2 * 4099 * 2.0 ** -53 * (np.abs(a) @ np.abs(b))).all()
    cap.close()


# A stream's first run under a relaxed capture gets the scratch it needs, for two
# key ranges, and no workspace for eight; a later run asks for that again, and
# the graph keeps its own.
def test_workspace_after_a_captured_first_run(hip):
    q, k, bias = operands(1, 2048, 128)
    art, bufs = built(hip, 1, 2048, 128), device(q, k, bias)
    out, eager, fresh = (DeviceBuffer(2048 * 2048, "f32") for _ in range(3))
    built(hip, 1, 2048, 128).run_device({**bufs, 3: fresh})
    cap = _Capture(mode=2)
    with cap as stream:
        art.run_device({**bufs, 3: out}, stream=stream, sync=False)
    for _ in range(3):
        cap.replay()
        check(out.to_numpy(), q, k, bias)
        art.run_device({**bufs, 3: eager}, stream=cap.stream.value, sync=False)
        cap("hipStreamSynchronize", cap.stream)
        assert np.array_equal(eager.to_numpy(), fresh.to_numpy())
    assert not np.array_equal(out.to_numpy(), fresh.to_numpy())     # two ranges add up in another order
    cap.close()
