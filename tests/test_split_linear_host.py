"""What the split products refuse before anything is launched."""
import ctypes

import pytest

from quick_ssm_amd import _lib

MANY = 5


class _Call(ctypes.Structure):
    """qssm_split_gemm_call of include/quick_ssm_hip.h."""

    _fields_ = [
        ("a", ctypes.c_void_p * MANY), ("b", ctypes.c_void_p * MANY), ("c", ctypes.c_void_p * MANY),
        ("bias", ctypes.c_void_p * MANY), ("amax_a", ctypes.c_void_p * MANY), ("amax_b", ctypes.c_void_p * MANY),
        ("lda", ctypes.c_int64), ("ldb", ctypes.c_int64), ("ldc", ctypes.c_int64),
        *((name, ctypes.c_int32) for name in ("M", "N", "K", "batch", "segments", "splits", "a_kstrided", "b_kstrided",
                                              "parts_a", "parts_b")),
        ("partial", ctypes.c_void_p), ("partial_floats", ctypes.c_uint64),
    ]


@pytest.mark.parametrize("m,n", [(2 ** 31 - 1, 4), (2 ** 31 - 256, 4), (4, 2 ** 31 - 4), (4, 2 ** 31 - 128)])
def test_sizes_whose_last_tile_ends_beyond_32_bits_are_refused(m, n):
    # The kernel's row and column numbers run to the end of the last tile of 256 x 128 in 32 bits; the addresses here
    # are never looked at, because the call ends before a launch.
    lib = _lib.load()
    lib.qssm_split_gemm.restype = ctypes.c_int
    lib.qssm_split_gemm.argtypes = [ctypes.POINTER(_Call), ctypes.c_void_p]
    call = _Call(M=m, N=n, K=4, lda=4, ldb=4, ldc=-(-n // 4) * 4, batch=1, segments=1, splits=1, parts_a=1, parts_b=1)
    for field in ("a", "b", "c", "amax_a", "amax_b"):
        getattr(call, field)[0] = 4096
    assert lib.qssm_split_gemm(ctypes.byref(call), None) == _lib.QSSM_EINVAL
