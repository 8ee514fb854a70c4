"""The split products without a GPU: what they refuse before anything is launched, and the arithmetic they rest on."""
import ctypes

import pytest
import torch

from quick_ssm_amd import _lib

MANY = 5


class _Call(ctypes.Structure):
    """qssm_gemm_f32_call of include/quick_ssm_hip.h."""

    _fields_ = [
        ("a", ctypes.c_void_p * MANY), ("b", ctypes.c_void_p * MANY), ("c", ctypes.c_void_p * MANY),
        ("bias", ctypes.c_void_p * MANY),
        ("lda", ctypes.c_int64), ("ldb", ctypes.c_int64), ("ldc", ctypes.c_int64),
        *((name, ctypes.c_int32) for name in ("M", "N", "K", "batch", "segments", "splits", "a_kstrided", "b_kstrided")),
        ("partial", ctypes.c_void_p), ("partial_floats", ctypes.c_uint64),
    ]


@pytest.mark.parametrize("m,n", [(2 ** 31 - 1, 4), (2 ** 31 - 128, 4), (4, 2 ** 31 - 4), (4, 2 ** 31 - 128)])
def test_sizes_whose_last_tile_ends_beyond_32_bits_are_refused(m, n):
    # The kernel's row and column numbers run to the end of the last tile of 128 x 128 in 32 bits; the addresses here
    # are never looked at, because the call ends before a launch.
    lib = _lib.load()
    lib.qssm_gemm_f32.restype = ctypes.c_int
    lib.qssm_gemm_f32.argtypes = [ctypes.POINTER(_Call), ctypes.c_void_p]
    call = _Call(M=m, N=n, K=4, lda=4, ldb=4, ldc=-(-n // 4) * 4, batch=1, segments=1, splits=1)
    for field in ("a", "b", "c"):
        getattr(call, field)[0] = 4096
    assert lib.qssm_gemm_f32(ctypes.byref(call), None) == _lib.QSSM_EINVAL


def _parts(x):
    """The three bf16 values an element is split into, as float32."""
    out = []
    for _ in range(3):
        out.append(x.bfloat16().float())
        x = x - out[-1]
    return out


def test_three_bf16_parts_hold_every_bit_and_six_products_all_but_the_last():
    # What csrc/gemm_split.hip rests on.  Every fp32 number below 2^111, subnormals included, is exactly the sum of its
    # scaled parts; and what the six products leave out of a pair is below 2^-24 of it.
    bits = torch.randint(0, 1 << 31, (1 << 20,), generator=torch.Generator().manual_seed(1))
    x = torch.cat((bits.int(), torch.tensor([0, 1, 3, 0x7FFFFF, 0x800000, 0x800001, (127 + 111 << 23) - 1], dtype=torch.int32)))
    x = x.view(torch.float32)
    x = x[x.abs() < 2.0 ** 111]
    assert x.numel() > 1 << 19
    # (bf16's own smallest numbers are 2^-133; the scaled numbers' last bits are at or above that)
    total = sum(p.double() for p in _parts(x * 2.0 ** 16))
    assert torch.equal(total * 2.0 ** -16, x.double())
    gen = torch.Generator().manual_seed(2)
    a, b = (torch.randn(1 << 20, generator=gen) for _ in range(2))
    pa, pb = _parts(a), _parts(b)
    kept = sum(pa[i].double() * pb[j].double() for i, j in ((2, 0), (0, 2), (1, 1), (1, 0), (0, 1), (0, 0)))
    exact = a.double() * b.double()
    assert bool(((kept - exact).abs() <= 2.0 ** -24 * exact.abs()).all())


@pytest.mark.parametrize("n,k,many", [(8, 8, 1), (64, 64, 1), (80, 16, 1), (320, 64, 1), (64, 64, 5), (128, 128, 1), (640, 128, 1), (96, 96, 5)])
def test_scratch_for_a_packed_operand_is_bounded_by_the_operands(n, k, many):
    # Weight gradients [n, k] over many rows: an operand is packed in whole tiles of 256 columns, however narrow it is.
    lib = _lib.load()
    nbytes = ctypes.c_uint64()
    for rows in (8192, 32768, 262144, 1 << 20, 1 << 24):
        call = _Call(M=n, N=k, K=rows, lda=n, ldb=k, ldc=k, batch=many, segments=1, splits=1, a_kstrided=1, b_kstrided=1)
        for i in range(many):
            call.a[i], call.b[i], call.c[i] = 4096 * (2 + i), 4096, 8192
        _lib.check(lib.qssm_gemm_f32_packed_plan(ctypes.byref(call), ctypes.byref(nbytes)))
        assert nbytes.value <= 2 * 4 * rows * (n * many + k)
        assert 1 <= call.splits <= 64 and call.splits * n * k * many * 4 <= max(1 << 22, 4 * rows * (n * many + k))
