"""Products too large for one grid of the tiled kernels: HIP launches fewer than
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
