"""Work too large for one grid of the tiled kernels: HIP launches fewer than
2^32 threads, and the kernel that is chosen stays below (no device needed)."""
import ctypes

import pytest

from mlk2_amd.backend import DTYPE_CODE, lib


class _Gemm(ctypes.Structure):
    """mlkd_gemm of csrc/device_abi.h."""
    _fields_ = [("a", ctypes.c_void_p), ("b", ctypes.c_void_p), ("c", ctypes.c_void_p),
                ("a_dtype", ctypes.c_int32), ("b_dtype", ctypes.c_int32), ("c_dtype", ctypes.c_int32),
                ("accumulate", ctypes.c_int32), ("m", ctypes.c_int64), ("n", ctypes.c_int64), ("k", ctypes.c_int64),
                ("lda", ctypes.c_int64), ("ldb", ctypes.c_int64), ("ldc", ctypes.c_int64), ("variant", ctypes.c_int32),
                ("skip_zero_a", ctypes.c_int32), ("pad_", ctypes.c_int32), ("work", ctypes.c_void_p),
                ("work_bytes", ctypes.c_int64)]


# f32 C on 64 x 64 tiles of 512 threads: 2^23 of them, from 137 GB on, are too many.
@pytest.mark.parametrize("m,n,ragged", [(2000, 2001, True), (185300, 185301, True), (185409, 185409, False),
                                        (200001, 200002, False)])
@pytest.mark.parametrize("k", [64, 100])
def test_f32_products_past_one_grid(m, n, k, ragged):
    L = lib()
    L.mlkd_gemm_kernel_name.restype = ctypes.c_char_p
    L.mlkd_gemm_pad_bytes.restype = ctypes.c_int64
    f32 = DTYPE_CODE["f32"]
    p = _Gemm(1 << 20, 2 << 20, 3 << 20, f32, f32, f32, 0, m, n, k, k, n, n, -1, 0)
    p.work, p.work_bytes = 4 << 20, L.mlkd_gemm_pad_bytes(ctypes.byref(p))
    name = L.mlkd_gemm_kernel_name(ctypes.byref(p)).decode()
    rows, cols = ctypes.c_int64(), ctypes.c_int64()
    L.mlkd_gemm_tile(ctypes.byref(p), ctypes.byref(rows), ctypes.byref(cols))
    assert (rows.value, cols.value) == (64, 64)
    tiles = -(-m // 64) * -(-n // 64)
    if ragged:
        assert name == "gemmF32Dma<false>" and tiles * 512 < 1 << 32
    else:
        # The direct kernel: one wave to a tile where there are 2048 tiles and more.
        assert name == "gemmGeneral<float>" and tiles * 64 < 1 << 32


class _Score(ctypes.Structure):
    """mlkd_score_softmax of csrc/device_abi.h."""
    _fields_ = [("q", ctypes.c_void_p), ("k", ctypes.c_void_p), ("bias", ctypes.c_void_p), ("s", ctypes.c_void_p),
                ("qk_dtype", ctypes.c_int32), ("bias_dtype", ctypes.c_int32), ("s_dtype", ctypes.c_int32),
                ("variant", ctypes.c_int32), ("batch", ctypes.c_int64), ("seq", ctypes.c_int64), ("dim", ctypes.c_int64),
                ("div", ctypes.c_double), ("scratch", ctypes.c_void_p), ("scratch_bytes", ctypes.c_int64),
                ("work", ctypes.c_void_p), ("work_bytes", ctypes.c_int64)]


# Two passes of 256 threads to a key range of 128 query rows, however short the
# sequence: 2^24 workgroups are too many (1 key: operands of 4 GiB each).
@pytest.mark.parametrize("batch,seq,ranges", [((1 << 24) - 1, 1, 1), (1 << 24, 1, 0), (1 << 24, 7, 0), (1 << 25, 1, 0),
                                              (1 << 21, 128, 1), ((1 << 22) - 1, 256, 2), (1 << 22, 256, 0)])
def test_score_batches_past_one_grid(batch, seq, ranges):
    L = lib()
    L.mlkd_score_pad_bytes.restype = L.mlkd_score_scratch_bytes.restype = ctypes.c_int64
    L.mlkd_score_kernel_names.restype = ctypes.c_char_p
    f16, f32 = DTYPE_CODE["f16"], DTYPE_CODE["f32"]
    p = _Score(1 << 20, 2 << 20, 3 << 20, 4 << 20, f16, f32, f32, -1, batch, seq, 128, 8.0)
    pad, need = L.mlkd_score_pad_bytes(ctypes.byref(p)), L.mlkd_score_scratch_bytes(ctypes.byref(p))
    p.work = p.scratch = 5 << 20
    p.work_bytes = p.scratch_bytes = max(pad, need)
    names = L.mlkd_score_kernel_names(ctypes.byref(p)).decode()
    assert L.mlkd_score_ranges(ctypes.byref(p)) == ranges
    if ranges:
        assert names == "scoreStatsQ+scoreStoreQ" and batch * -(-seq // 128) * ranges * 256 < 1 << 32
    else:
        assert pad == need == 0 and names.startswith("scoresF16" if seq % 128 == 0 else "scoresGeneral")
